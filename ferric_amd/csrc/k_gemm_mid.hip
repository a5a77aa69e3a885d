// K1 projections of mid-sized batches (a prompt of some hundred rows, or a
// narrow weight): too few 256 x 256 blocks for the 256 CUs, too many rows to
// stream the weight once per row chunk. bf16 MFMA
// (v_mfma_f32_32x32x16_bf16), FP32 accumulation.
//
// A workgroup owns a block of 32 TN weight rows x 32 TM activation rows and
// its waves split k: wave w takes k-blocks w, w + WAVES, ... and accumulates
// the whole block over them, so the k loop has no LDS traffic and no
// barrier; every operand goes from its tile order (common.hpp) straight into
// registers, D half-k-block stages deep. At the end the waves' partial blocks
// are added in wave order through LDS, 32 activation rows at a time, where
// the epilogue also gets its row-contiguous stores. The sum over k is a
// reassociation of the serial order, as in the other projection kernels,
// fixed by the launch shape.
//
// What bounds it: the operands, read from L2 (2 (TN + TM) KiB per k-block and
// workgroup). Launches of 512 and more blocks on the models' weights read them
// at 15 to 17 TB/s over all CUs in the median of each shape (128 x 128 blocks:
// 11.6, with 8 us of reduction and epilogue), 24 at most, with and without the
// MFMAs and at 3 to 7 stages in flight. So large blocks read less and small ones
// fill the CUs; gemm_mid_cost weighs the two.
// Measured against the 256 x 256-block kernel (us per launch, cold weights):
//   777 rows: O 4096 x 4096 87 -> 38, down 4096 x 12288 225 -> 101
//   512 rows: O 1024 x 2048 48 -> 7.4, down 1024 x 3072 64 -> 10.0, gate/up 6144 x 1024 30 -> 12.2
//   288 rows: O 4096 x 4096 87 -> 28
//   48 rows: down 4096 x 12288 56 (the weight-streaming kernel over row chunks) -> 32
//
// A 32x32x16 operand (lane l: row l % 32, columns 8 (l / 32) .. + 7) is half
// a k-block of two adjacent 16-row tiles: in-tile lanes l % 16 + 16 (l / 32)
// (+ 32 for the second half) of tile (l / 16) % 2, so a load is four
// contiguous 256-byte runs.
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "../../include/ferric_hip.h"

namespace fh {

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ bf16x8 b8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// Calls f(std::integral_constant<int, I>) for I = B .. E - 1, unrolled at compile time.
template <int B, int E, class F>
__device__ __forceinline__ void mid_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    mid_for<B + 1, E>(f);
  }
}

// From this k on the 8 tiles that a 128-row block has per k-block span 4 GiB.
constexpr uint32_t kMidFarK = 1u << 24;

// The QKV projection with QK-norm, RoPE and the KV append in its epilogue
// (TN = 4: a workgroup's columns are one head).
constexpr int kMidEpiQkvRope = 16;

// kFar: 64-bit operand addresses (global loads) for a k whose weight rows the
// buffer loads' 32-bit offsets do not reach (kMidFarK).
template <int TN, int TM, int WAVES, int D, int OCC, int EPI, bool kFar>
__global__ __launch_bounds__(WAVES * 64, OCC) void gemm_mid_kernel(const uint16_t* __restrict__ xt,
                                                                   const uint16_t* __restrict__ w, uint32_t m,
                                                                   uint32_t mtiles, uint32_t kb_count,
                                                                   const uint16_t* residual, void* out, uint32_t ldo,
                                                                   const QkvRopeArgs qa, uint32_t* err) {
  constexpr int kN = 32 * TN, kPitch = kN + 4, kThreads = WAVES * 64;
  constexpr size_t kRedBytes = sizeof(float) * WAVES * 32 * kPitch;
  constexpr size_t kStageBytes = EPI == kMidEpiQkvRope ? 4ull * 32 * TM * kQkPitch : 0;
  constexpr int kQkRows = 32 * TM / WAVES;  // rows a wave of the fused QKV epilogue takes
  static_assert(EPI != kMidEpiQkvRope || (TN == 4 && kQkRows % 8 == 0 && kQkRows <= 64), "one head per workgroup");
  static_assert(kRedBytes >= kStageBytes, "the staged head rows reuse the reduction's LDS");
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[kRedBytes];
  auto& red = *reinterpret_cast<float(*)[WAVES][32][kPitch]>(lds_raw);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Block order by XCD (workgroups go to the 8 XCDs round-robin): XCD j takes
  // n-blocks j, j + 8, ... and walks all m-blocks of each, so a weight tile
  // is fetched into one XCD's L2 only. N-blocks past the last multiple of 8
  // keep their m-blocks consecutive in dispatch order.
  const uint32_t NB = gridDim.x, MB = gridDim.y, N8 = NB & ~7u, b = blockIdx.x + NB * blockIdx.y;
  uint32_t gx, gy;
  if (b < N8 * MB) {
    const uint32_t r = b >> 3;
    gy = r % MB;
    gx = (r / MB) * 8 + (b & 7u);
  } else {
    const uint32_t t = b - N8 * MB;
    gx = N8 + t / MB;
    gy = t % MB;
  }
  // The fused QKV epilogue's row lookups (position, page, slot) are requested
  // now and used after the k loop.
  QkvRowSlot row_slot{0u, 0u, false};
  if constexpr (EPI == kMidEpiQkvRope) {
    const uint32_t row = gy * 32 * TM + wave * kQkRows + lane;
    if (lane < kQkRows && row < m) row_slot = qkv_row_slot(row, qa);
  }
  const uint32_t kb_n = kb_count > (uint32_t)wave ? (kb_count - wave + WAVES - 1) / WAVES : 0u;  // k-blocks of this wave
  f32x16 acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  if (kb_n > 0) {
    // Buffer descriptors: the block's weight rows from k-block `wave` on
    // (32-bit offsets: k < kMidFarK), and one k-block of its activation rows.
    const uint64_t w0 = ((uint64_t)gx * 2 * TN * kb_count + wave) * 512, x0 = ((uint64_t)wave * mtiles + gy * 2 * TM) * 512;
    auto wrs = __builtin_amdgcn_make_buffer_rsrc((void*)(w + w0), 0, (2u * TN * kb_count - wave) * 1024u, 0x00020000);
    const uint32_t in_tile = (lane & 15) + 16 * (lane >> 5), second = (lane >> 4) & 1;
    const uint32_t wofs = (second * kb_count * 64 + in_tile) * 16, xofs = (second * 64 + in_tile) * 16;
    const uint32_t wpair = kb_count * 2048u;
    const u32x4* wfar = reinterpret_cast<const u32x4*>(w + w0) + (uint64_t)second * kb_count * 64 + in_tile;
    const u32x4* xfar = reinterpret_cast<const u32x4*>(xt + x0) + second * 64 + in_tile;
    // Stage: the operands of half a k-block.
    u32x4 wr[D][TN], xr[D][TM];
    const uint32_t halves = 2 * kb_n;
    auto load = [&](auto slot_c, uint32_t hk) {
      constexpr int S = decltype(slot_c)::value;
      const uint32_t q = min(hk, halves - 1), kk = (q >> 1) * WAVES, half = (q & 1u) * 512;
      if constexpr (kFar) {
#pragma unroll
        for (int i = 0; i < TN; ++i) wr[S][i] = wfar[((uint64_t)kk + 2ull * i * kb_count) * 64 + half / 16];
#pragma unroll
        for (int j = 0; j < TM; ++j) xr[S][j] = xfar[(uint64_t)kk * mtiles * 64 + half / 16 + j * 128];
        return;
      }
      const uint32_t ws = kk * 1024 + half;
      auto xrs = __builtin_amdgcn_make_buffer_rsrc((void*)(xt + x0 + (uint64_t)kk * mtiles * 512), 0, 2 * TM * 1024u, 0x00020000);
#pragma unroll
      for (int i = 0; i < TN; ++i)
        wr[S][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrs, wofs, ws + i * wpair, 0));
#pragma unroll
      for (int j = 0; j < TM; ++j)
        xr[S][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xrs, xofs, half + j * 2048, 0));
    };
    auto compute = [&](auto slot_c) {
      constexpr int S = decltype(slot_c)::value;
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b8(wr[S][i]), b8(xr[S][j]), acc[i][j], 0, 0, 0);
    };
    mid_for<0, D - 1>([&](auto s) { load(s, decltype(s)::value); });
    uint32_t hk = 0;
    for (; hk + D <= halves; hk += D)
      mid_for<0, D>([&](auto s) {
        constexpr int S = decltype(s)::value;
        load(std::integral_constant<int, (S + D - 1) % D>{}, hk + S + D - 1);
        __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the MFMAs
        compute(s);
        __builtin_amdgcn_sched_barrier(0);
      });
    mid_for<0, D - 1>([&](auto s) {
      if (hk + decltype(s)::value < halves) compute(s);
    });
  }

  // D layout: lane l, element e holds weight row 8 (e / 4) + 4 (l / 32) + e % 4
  // and activation row l % 32 of the 32 x 32 block.
  const uint32_t hi = lane >> 5, c = lane & 31;
  const uint32_t n0 = gx * kN;
  constexpr int kSteps = (32 * kN / 4 + kThreads - 1) / kThreads;
  bool bad = false;
  // The residual is requested before the reduction (out may alias it, so the
  // compiler cannot move a load over a store: one by one they would cost a
  // memory round trip each).
  constexpr bool kRes = EPI == FH_EPI_RESIDUAL;
  uint2 rv[kRes ? TM : 1][kRes ? kSteps : 1];
  if constexpr (kRes) {
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        const int idx = min((int)threadIdx.x + s * kThreads, 32 * kN / 4 - 1);
        const uint32_t row = min((gy * TM + j) * 32 + idx / (kN / 4), m - 1);
        rv[j][s] = *reinterpret_cast<const uint2*>(residual + (uint64_t)row * ldo + n0 + idx % (kN / 4) * 4);
      }
  }
  uint2 packed[EPI == kMidEpiQkvRope ? TM : 1][EPI == kMidEpiQkvRope ? kSteps : 1];
  mid_for<0, TM>([&](auto j_c) {
    constexpr int j = decltype(j_c)::value;
    if constexpr (j > 0) __syncthreads();
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *reinterpret_cast<f32x4*>(&red[wave][c][32 * i + 8 * e + 4 * hi]) =
            f32x4{acc[i][j][4 * e], acc[i][j][4 * e + 1], acc[i][j][4 * e + 2], acc[i][j][4 * e + 3]};
    __syncthreads();
    // Four consecutive columns of one row, the waves' partials in wave order.
    auto sum4 = [&](int r, int col) {
      f32x4 v = *reinterpret_cast<const f32x4*>(&red[0][r][col]);
#pragma unroll
      for (int q = 1; q < WAVES; ++q) {
        const f32x4 p = *reinterpret_cast<const f32x4*>(&red[q][r][col]);
        v = f32x4{v[0] + p[0], v[1] + p[1], v[2] + p[2], v[3] + p[3]};
      }
      return v;
    };
    const uint32_t row0 = (gy * TM + j) * 32;
    if constexpr (EPI == FH_EPI_SWIGLU) {
      // Column group i holds a gate tile (16 columns) and its up tile. Threads
      // walk the output in tile order: 4-column half, row, 8-column group, row tile.
      for (int idx = threadIdx.x; idx < 32 * kN / 8; idx += kThreads) {
        const int half = idx & 1, r = (idx >> 1) & 15, g = (idx >> 5) % (2 * TN), mt = (idx >> 5) / (2 * TN);
        const uint32_t row = row0 + 16 * mt + r;
        if (row >= m) continue;
        const int col = 32 * (g >> 1) + 8 * (g & 1) + 4 * half;
        const f32x4 gate = sum4(16 * mt + r, col), up = sum4(16 * mt + r, col + 16);
        uint32_t y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = swiglu_bf16(round_bf16(gate[e]), round_bf16(up[e]), bad);
        *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out) + act_offset_m(row, n0 / 2 + 8 * g + 4 * half, mtiles)) =
            make_uint2(y[0] | (y[1] << 16), y[2] | (y[3] << 16));
      }
    } else {
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        const int idx = threadIdx.x + s * kThreads;
        if (32 * kN / 4 % kThreads != 0 && idx >= 32 * kN / 4) break;
        const int r = idx / (kN / 4), col = idx % (kN / 4) * 4;
        const uint32_t row = row0 + r;
        const f32x4 v = sum4(r, col);
        if constexpr (EPI == kMidEpiQkvRope) {
          packed[j][s] = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
        } else if (row < m) {
          const uint64_t o = (uint64_t)row * ldo + n0 + col;
          if constexpr (EPI == FH_EPI_F32) {
            *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(out) + o) = v;
          } else if constexpr (EPI == FH_EPI_BF16) {
            *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out) + o) =
                make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
          } else {
            const uint2 r0 = rv[j][s];
            *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out) + o) =
                make_uint2(pack_bf16x2((0.0f + v[0]) + lo_bf16(r0.x), (0.0f + v[1]) + hi_bf16(r0.x)),
                           pack_bf16x2((0.0f + v[2]) + lo_bf16(r0.y), (0.0f + v[3]) + hi_bf16(r0.y)));
          }
        }
      }
    }
  });
  if constexpr (EPI == FH_EPI_SWIGLU) {
    if (bad) raise_error(err, ERR_NONFINITE);
  }
  if constexpr (EPI == kMidEpiQkvRope) {
    // The head's rows staged as bf16 (the projection's rounding), then each
    // wave runs the QK-norm, RoPE and KV append of its share (qk_head.hpp).
    uint32_t* rows_lds = reinterpret_cast<uint32_t*>(lds_raw);
    __syncthreads();  // every wave is done reading the reduction's LDS
    mid_for<0, TM>([&](auto j_c) {
      constexpr int j = decltype(j_c)::value;
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        const int idx = threadIdx.x + s * kThreads;
        *reinterpret_cast<uint2*>(rows_lds + (32 * j + idx / (kN / 4)) * kQkPitch + idx % (kN / 4) * 2) = packed[j][s];
      }
    });
    __syncthreads();
    qknorm_rope_kv_wave<kQkRows>(rows_lds + wave * kQkRows * kQkPitch, gy * 32 * TM + wave * kQkRows, m, gx, qa, row_slot);
  }
}

// Block shapes: 32 tn weight rows x 32 tm activation rows, and what
// mid_cost needs of each: the operand GB/s of a CU running such blocks alone,
// microseconds per launch and per 256 blocks around the k loop (prologue,
// reduction, epilogue), and the same two where k is so short that nothing else
// is left.
struct MidShape {
  uint32_t tn, tm;
  float cu_gbs, launch_us, round_us, least_us, least_round_us;
};
constexpr MidShape kMidShapes[] = {{4, 4, 69.0f, 0.55f, 6.84f, 11.22f, 3.58f}, {4, 2, 73.1f, 1.92f, 0.62f, 6.69f, 1.91f},
                                    {2, 4, 83.1f, 2.59f, 1.45f, 4.82f, 1.09f}, {2, 2, 75.9f, 1.47f, 0.02f, 4.00f, 0.80f},
                                    {1, 2, 83.1f, 2.45f, 0.26f, 3.72f, 0.64f}, {1, 1, 64.0f, 3.08f, 0.19f, 2.94f, 0.84f}};
// Microseconds that the SwiGLU and the QK-norm epilogues take longer, per 256
// blocks of 4 32 x 32 outputs.
constexpr float kMidSwigluUs = 0.14f, kMidQkvUs = 0.40f;

// Estimated microseconds of one launch: the operand bytes of all blocks at
// 18.2 TB/s, but no less than those of the blocks one CU runs at its own
// rate, plus the shape's overheads; and no less than the launch takes at a k
// of a few k-blocks. Its constants and those of the other two kernels'
// estimates (gemm_band_cost, block_cost) are fitted together to the times of
// every form at 3261 launches: 33 to 8192 rows of the Qwen3 projections, their
// fused QKV form, other wide weights and weights of 128 to 512 columns at k of
// 1024 to 12288, and 128 to 16512 columns at k of 32 to 768, with all
// epilogues. The estimate picks a form that is slower than the fastest by (mean,
// most): Qwen3 projections 1.8 %, 25 % (64 x 4096 x 1024 6.0 us, 4.8 possible); fused
// QKV 0.8 %, 21 %; other wide weights 1.9 %, 27 %; narrow weights 3.9 %, 69 % (2048 x
// 256 x 12288 58 us, 34.5 possible); k up to 768 3.6 %, 55 %. At k of 1024 and more
// it is never more than 3 % slower than the 256 x 256 blocks alone. (Constants
// fitted to 296 launches of the Qwen3 projections only, without the least time
// and the epilogues' own, took 128 x 128 blocks for every k of up to 128: 96 x
// 128 x 64 5.9 us, now 2.9, 4.8 with the weight stream before these blocks. Where
// their choice was no slower than before these blocks, the fit keeps it for the
// Qwen3 projections of up to 256 rows.)
float mid_cost(const MidShape& s, uint32_t m, uint32_t n, uint32_t k, uint32_t epilogue, bool fused_qkv) {
  const float rounds = (float)(n / (32 * s.tn)) * ((m + 32 * s.tm - 1) / (32 * s.tm)) / 256.f;
  const float block_kb = 2.048f * (s.tn + s.tm) * (k / 32);  // operand kilobytes of a block
  const float all = rounds * 256.f * block_kb / 18200.f;
  const float cu = ceilf(rounds) * block_kb / s.cu_gbs;
  const float more = (fused_qkv ? kMidQkvUs : epilogue == FH_EPI_SWIGLU ? kMidSwigluUs : 0.f) * (s.tn * s.tm / 4.f);
  return fmaxf(s.least_us + rounds * (s.least_round_us + more),
               s.launch_us + rounds * (s.round_us + more) + fmaxf(all, cu));
}

bool mid_pick(uint32_t m, uint32_t n, uint32_t k, uint32_t epilogue, bool fused_qkv, MidShape* pick, float* cost) {
  bool found = false;
  for (const MidShape& s : kMidShapes) {
    if (n % (32 * s.tn) != 0 || (fused_qkv && s.tn != 4) || (k >= kMidFarK && s.tn * s.tm != 1)) continue;
    const float c = mid_cost(s, m, n, k, epilogue, fused_qkv);
    if (!found || c < *cost) {
      *pick = s;
      *cost = c;
      found = true;
    }
  }
  return found;
}

template <int TN, int TM, int WAVES, int D, int OCC, int EPI, bool kFar = false>
void launch_mid_variant(const uint16_t* xt, const uint16_t* w, uint32_t m, uint32_t n, uint32_t k,
                        const uint16_t* residual, void* out, uint32_t ldo, const QkvRopeArgs& qa, uint32_t* err,
                        hipStream_t s) {
  hipLaunchKernelGGL((gemm_mid_kernel<TN, TM, WAVES, D, OCC, EPI, kFar>), dim3(n / (32 * TN), (m + 32 * TM - 1) / (32 * TM)),
                     dim3(WAVES * 64), 0, s, xt, w, m, act_mtiles(m), k / 32, residual, out, ldo, qa, err);
}

// Waves per workgroup, stages and workgroups per CU of each shape: 4 waves
// while the accumulators (16 TN TM registers) leave no room for more, 8 for
// the small blocks, whose waves would else have too little in flight.
template <int EPI>
hipError_t launch_mid_shape(MidShape v, const uint16_t* xt, const uint16_t* w, uint32_t m, uint32_t n, uint32_t k,
                            const uint16_t* residual, void* out, uint32_t ldo, const QkvRopeArgs& qa, uint32_t* err,
                            hipStream_t s) {
#define FH_MID(TN_, TM_, WAVES_, D_, OCC_) \
  launch_mid_variant<TN_, TM_, WAVES_, D_, OCC_, EPI>(xt, w, m, n, k, residual, out, ldo, qa, err, s)
  if (k >= kMidFarK) {
    if constexpr (EPI == kMidEpiQkvRope) return hipErrorInvalidValue;
    else launch_mid_variant<1, 1, 8, 12, 2, EPI, true>(xt, w, m, n, k, residual, out, ldo, qa, err, s);
  } else if (v.tn == 4 && v.tm == 4) {
    FH_MID(4, 4, 4, 4, 1);
  } else if (v.tn == 4) {
    FH_MID(4, 2, 4, 4, 2);
  } else if constexpr (EPI != kMidEpiQkvRope) {
    if (v.tn == 2 && v.tm == 4)
      FH_MID(2, 4, 4, 4, 2);
    else if (v.tn == 2)
      FH_MID(2, 2, 4, 6, 2);
    else if (v.tm == 2)
      FH_MID(1, 2, 8, 6, 2);
    else
      FH_MID(1, 1, 8, 12, 2);
  } else {
    return hipErrorInvalidValue;
  }
#undef FH_MID
  return hipGetLastError();
}

}  // namespace

float gemm_mid_cost(uint32_t m, uint32_t n, uint32_t k, uint32_t epilogue, bool fused_qkv) {
  MidShape v{};
  float cost = 0.f;
  return m > kMaxRows && n % 32 == 0 && k % 32 == 0 && k > 0 && mid_pick(m, n, k, epilogue, fused_qkv, &v, &cost)
             ? cost
             : -1.f;
}

uint32_t gemm_mid_block(uint32_t m, uint32_t n, uint32_t k, uint32_t epilogue, bool fused_qkv) {
  MidShape v{};
  float cost = 0.f;
  return mid_pick(m, n, k, epilogue, fused_qkv, &v, &cost) ? (32 * v.tm) << 16 | 32 * v.tn : 0u;
}

hipError_t launch_gemm_mid(const uint16_t* x_tiled, const uint16_t* w_tiled, uint32_t m, uint32_t n, uint32_t k,
                           uint32_t epilogue, const uint16_t* residual, void* out, uint32_t ldo, uint32_t* err,
                           hipStream_t s) {
  MidShape v{};
  float cost = 0.f;
  if (m <= kMaxRows || n % 32 != 0 || k % 32 != 0 || k == 0 || !mid_pick(m, n, k, epilogue, false, &v, &cost))
    return hipErrorInvalidValue;
  const QkvRopeArgs none{};
#define FH_MID_EPI(E) \
  case E: return launch_mid_shape<E>(v, x_tiled, w_tiled, m, n, k, residual, out, ldo, none, err, s)
  switch (epilogue) {
    FH_MID_EPI(FH_EPI_BF16);
    FH_MID_EPI(FH_EPI_RESIDUAL);
    FH_MID_EPI(FH_EPI_SWIGLU);
    FH_MID_EPI(FH_EPI_F32);
    default: return hipErrorInvalidValue;
  }
#undef FH_MID_EPI
}

hipError_t launch_gemm_mid_qkv_rope(const uint16_t* x_tiled, const uint16_t* w_tiled, uint32_t m, uint32_t n,
                                    uint32_t k, const QkvRopeArgs& qa, hipStream_t s) {
  MidShape v{};
  float cost = 0.f;
  if (m <= kMaxRows || n != (qa.qh + 2 * qa.kvh) * 128 || k % 32 != 0 || k == 0 || !mid_pick(m, n, k, FH_EPI_BF16, true, &v, &cost))
    return hipErrorInvalidValue;
  return launch_mid_shape<kMidEpiQkvRope>(v, x_tiled, w_tiled, m, n, k, nullptr, nullptr, 0u, qa, nullptr, s);
}

}  // namespace fh
