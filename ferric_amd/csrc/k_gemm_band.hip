// K1 projections for prefill chunks of 256-row x 128-column blocks: bf16
// MFMA (v_mfma_f32_32x32x16_bf16), FP32 accumulation. launch_gemm_large
// chooses between these blocks, the smaller ones of k_gemm_mid.hip and the
// 256 x 256 ones of k_gemm_large.hip.
//
// Operands come from their tile orders (common.hpp): the weight in weight
// tile order and the activation in activation tile order with act_mtiles(m)
// row tiles. A workgroup has 4 waves of 64 rows each. Each k-block's 8 weight
// tiles are fetched global -> LDS directly (16 bytes per lane, the tile order
// itself) into an (LW + 1)-stage ring that all waves read; a wave's own 4
// activation tiles are read by no other wave and go straight into registers
// (an (LX + 1)-slot ring). A 32x32x16 operand is half a k-block of two
// adjacent 16-row tiles (lane l: in-tile lane l % 16 + 16 (l / 32), tile
// (l / 16) % 2). Two workgroups share a CU (128 accumulator registers, 72 KiB
// of LDS), so one's prologue and epilogue run beside the other's k loop.
//
// Both loads are buffer loads. With the weight fetch as a global load to LDS
// (a FLAT-encoded instruction) the compiler turns every later wait for an LDS
// read or a register load into a wait for all of them; with buffer loads its
// waits count only what must have arrived, so a wave's LDS reads stay three
// column groups ahead of their MFMAs, across the barrier as well.
//
// Epilogues (same rounding points as the decode kernel, no split-K here):
//   FH_EPI_BF16     out[m][n] = bf16(acc)
//   FH_EPI_RESIDUAL out[m][n] = bf16((0 + acc) + residual[m][n]) (may alias out)
//   FH_EPI_SWIGLU   act = swiglu(bf16(gate), bf16(up)) in activation tile order
//                   (gate/up tiles interleaved by the weight layout)
//   FH_EPI_F32      out[m][n] = acc (FP32 logits)
// The accumulators go through LDS 64 columns at a time, so that a store
// writes whole 128-byte lines of a row: straight from the MFMA layout a store
// touches 32 rows with 16 bytes each.
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "../../include/ferric_hip.h"

namespace fh {

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kBandWaves = 4;
constexpr int kBandCols = 128;
static_assert(kLargeBlockRows == 64 * kBandWaves, "64 rows per wave");

__device__ __forceinline__ bf16x8 b8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

constexpr unsigned band_wait_vm(unsigned n) { return (n & 15u) | ((n >> 4) << 14) | (7u << 4) | (15u << 8); }

// Calls f(std::integral_constant<int, I>) for I = B .. E - 1, unrolled at compile time.
template <int B, int E, class F>
__device__ __forceinline__ void band_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    band_for<B + 1, E>(f);
  }
}

__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// EPI == kBandEpiQkvRope (the QKV projection of a prefill chunk): 4 column groups
// are one head (128 columns) of the wave's 64 rows. The wave stages them in
// LDS as bf16 rows (the projection's rounding) and lane r runs the per-head
// QK-norm, RoPE and KV append of row r (qk_head.hpp), without the QKV output's
// round trip through HBM or a second launch.
constexpr int kBandEpiQkvRope = 16;
constexpr int kStagePitch = 68;  // floats per staged row of 64 columns

template <int EPI>
__global__ __launch_bounds__(64 * kBandWaves, 2) void gemm_band_kernel(const uint16_t* __restrict__ xt,
                                                                           const uint16_t* __restrict__ w, uint32_t m,
                                                                           uint32_t mtiles, uint32_t kb_count,
                                                                           const uint16_t* residual, void* out,
                                                                           uint32_t ldo, const QkvRopeArgs qa,
                                                                           uint32_t* err) {
  constexpr int CG = kBandCols / 32, LX = 4, LW = 8;
  constexpr int WT = 2 * CG;                      // weight tiles per k-block
  constexpr int WPW = WT / kBandWaves;           // of which each wave fetches this many
  constexpr int XPW = 4;                          // activation tiles per wave and k-block
  constexpr int WST = LW + 1, XS = LX + 1, R = 4;  // ring sizes; column groups of weight operands in registers
  static_assert(CG % R == 0, "a column group's register slot is the same in every k-block");
  // The wait before k-block kb counts per kind: direct-to-LDS loads (the
  // weight tiles) and register loads (the activation tiles) complete out of
  // order with respect to each other, only loads of one kind in issue order.
  // Needed are W(kb + 1) (its first column groups are read during kb) and
  // X(kb): if the first were outstanding, so would be the WPW (LW - 2) weight
  // loads after it, if the second, the XPW (LX - 1) activation loads after
  // it. At most the smaller count outstanding covers both.
  constexpr unsigned kWLater = WPW * (LW - 2), kXLater = XPW * (LX - 1);
  constexpr unsigned kInFlight = kWLater < kXLater ? kWLater : kXLater;
  static_assert(LW >= 2 && LX >= 1 && LW >= LX && WPW * (LW - 1) < 64, "vmcnt range");
  constexpr size_t kRingBytes = sizeof(u32x4) * WST * WT * 64;
  constexpr size_t kStageBytes =
      EPI == kBandEpiQkvRope ? 4ull * kBandWaves * 64 * kQkPitch : sizeof(float) * kBandWaves * 64 * kStagePitch;
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[kRingBytes > kStageBytes ? kRingBytes : kStageBytes];
  auto& wlds = *reinterpret_cast<u32x4(*)[WST][WT][64]>(lds_raw);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Block order by XCD: workgroups go to the 8 XCDs round-robin in dispatch
  // order, and each XCD has its own L2. With a multiple of 32 m-blocks XCD j
  // takes m-blocks j, j + 8, ... four at a time and walks all n-blocks with
  // them; else it takes n-blocks j, j + 8, ... and walks all m-blocks of each.
  const uint32_t NB = gridDim.x, MB = gridDim.y, b = blockIdx.x + NB * blockIdx.y;
  uint32_t gx, gy;
  if (MB % 32 == 0) {
    const uint32_t r = b >> 3;  // position within this XCD's share
    const uint32_t group = r / (4 * NB), within = r % (4 * NB);
    gy = (group * 4 + within % 4) * 8 + (b & 7u);
    gx = within / 4;
  } else if (b < (NB & ~7u) * MB) {
    const uint32_t r = b >> 3;
    gy = r % MB;
    gx = (r / MB) * 8 + (b & 7u);
  } else {
    const uint32_t t = b - (NB & ~7u) * MB;
    gx = (NB & ~7u) + t / MB;
    gy = t % MB;
  }
  const uint32_t bn = gx * WT, row0 = gy * kLargeBlockRows + wave * 64;  // first weight tile, this wave's first row
  const bool live = row0 < m;  // a wave whose rows are all padding only helps fetch the weights
  const uint32_t last = kb_count - 1;
  // The fused QKV epilogue's row lookups (position, page, slot) are
  // requested now and used after the k loop.
  QkvRowSlot row_slot{0u, 0u, false};
  if constexpr (EPI == kBandEpiQkvRope) {
    if (row0 + lane < m) row_slot = qkv_row_slot(row0 + lane, qa);
  }
  auto wrs = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (uint64_t)bn * kb_count * 512), 0, WT * kb_count * 1024u,
                                               0x00020000);
  auto fetch_w = [&](uint32_t kb) {
    const uint32_t off = min(kb, last) * 1024u + (uint32_t)(WPW * wave) * kb_count * 1024u;
#pragma unroll
    for (int t = 0; t < WPW; ++t)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          wrs, (__attribute__((address_space(3))) void*)&wlds[kb % WST][WPW * wave + t][0], 16, lane * 16,
          off + t * (kb_count * 1024u), 0, 0);
  };

  f32x16 acc[CG][2];
#pragma unroll
  for (int i = 0; i < CG; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  const uint32_t lofs = ((lane >> 4) & 1) * 64 + (lane & 15) + 16 * (lane >> 5);  // 16-byte units
  if (live) {
    const uint16_t* xw = xt + (uint64_t)row0 * 32;  // tiles row0 / 16 .. + 3 of k-block 0
    u32x4 xr[XS][XPW];                              // [2 m-group + half]
    auto load_x = [&](auto slot_c, uint32_t kb) {
      auto xrs = __builtin_amdgcn_make_buffer_rsrc((void*)(xw + (uint64_t)min(kb, last) * mtiles * 512), 0, XPW * 1024u,
                                                   0x00020000);
#pragma unroll
      for (int j = 0; j < XPW; ++j)
        xr[decltype(slot_c)::value][j] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(xrs, lofs * 16, (j >> 1) * 2048 + (j & 1) * 512, 0));
    };
    // Issue order per iteration j: W(j + LW), then X(j + LX); k-blocks past
    // the end are clamped to the last one, so the count of loads in flight is
    // the same at every iteration. The prologue issues in that same order.
    band_for<0, LW>([&](auto j_c) {
      constexpr int j = decltype(j_c)::value - LW;
      fetch_w(j + LW);
      if constexpr (j + LX >= 0) load_x(std::integral_constant<int, (j + LX) % XS>{}, j + LX);
    });
    u32x4 wv[R][2];
    const u32x4* wl = &wlds[0][0][0] + lofs;
    auto read_group = [&](auto slot_c, uint32_t stage, int g) {
#pragma unroll
      for (int h = 0; h < 2; ++h) wv[decltype(slot_c)::value][h] = wl[(stage * WT + 2 * g) * 64 + h * 32];
    };
    __builtin_amdgcn_s_waitcnt(band_wait_vm(WPW * (LW - 1)));
    __builtin_amdgcn_s_barrier();  // W(0) of every wave is in LDS
    band_for<0, R - 1>([&](auto g) { read_group(g, 0, decltype(g)::value); });
    auto step = [&](auto s_c, uint32_t kb) {
      constexpr int S = decltype(s_c)::value;
      __builtin_amdgcn_s_waitcnt(band_wait_vm(kInFlight));
      // W(kb + 1) of every wave is in LDS, and every wave is done reading
      // k-block kb - 1, whose stage the next fetch overwrites.
      __builtin_amdgcn_s_barrier();
      fetch_w(kb + LW);
      load_x(std::integral_constant<int, (S + LX) % XS>{}, kb + LX);
      const uint32_t st = kb % WST, st1 = (kb + 1) % WST;
      band_for<0, CG>([&](auto g_c) {
        constexpr int g = decltype(g_c)::value;
        constexpr int ahead = g + R - 1;
        if constexpr (ahead < CG)
          read_group(std::integral_constant<int, ahead % R>{}, st, ahead);
        else
          read_group(std::integral_constant<int, ahead % R>{}, st1, ahead - CG);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[g][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b8(wv[g % R][h]), b8(xr[S][2 * j + h]), acc[g][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);  // keeps the reads R - 1 groups ahead
      });
    };
    uint32_t kb = 0;
    for (; kb + XS <= kb_count; kb += XS)
      band_for<0, XS>([&](auto s_c) { step(s_c, kb + decltype(s_c)::value); });
    band_for<0, XS - 1>([&](auto s_c) {
      if (kb + decltype(s_c)::value < kb_count) step(s_c, kb + decltype(s_c)::value);
    });
  } else {
    band_for<0, LW>([&](auto j_c) { fetch_w(decltype(j_c)::value); });
    __builtin_amdgcn_s_waitcnt(band_wait_vm(WPW * (LW - 1)));
    __builtin_amdgcn_s_barrier();
    for (uint32_t kb = 0; kb < kb_count; ++kb) {
      __builtin_amdgcn_s_waitcnt(band_wait_vm(kWLater));
      __builtin_amdgcn_s_barrier();
      fetch_w(kb + LW);
    }
  }
  __builtin_amdgcn_s_waitcnt(band_wait_vm(0));  // the repeated loads past the end
  __syncthreads();  // every wave is done reading the weight ring, which the staging reuses
  if (!live) return;

  // D layout: lane l, element e holds weight row 8 (e / 4) + 4 (l / 32) + e % 4
  // and activation row l % 32 of a 32 x 32 block.
  const uint32_t hi = lane >> 5, c = lane & 31;
  if constexpr (EPI == kBandEpiQkvRope) {
    static_assert(CG % 4 == 0, "whole heads");
    uint32_t* rows_lds = reinterpret_cast<uint32_t*>(lds_raw) + (uint32_t)wave * 64 * kQkPitch;
    band_for<0, CG / 4>([&](auto h_c) {
      constexpr int head = decltype(h_c)::value;
      if constexpr (head > 0) wave_fence();
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const f32x16& a = acc[4 * head + i][j];
            *reinterpret_cast<uint2*>(rows_lds + (32 * j + c) * kQkPitch + 16 * i + 4 * e + 2 * hi) =
                make_uint2(pack_bf16x2(a[4 * e], a[4 * e + 1]), pack_bf16x2(a[4 * e + 2], a[4 * e + 3]));
          }
      wave_fence();
      qknorm_rope_kv_wave<64>(rows_lds, row0, m, gx * (CG / 4) + head, qa, row_slot);
    });
  } else {
    float* stage = reinterpret_cast<float*>(lds_raw) + (uint32_t)wave * 64 * kStagePitch;
    bool bad = false;
    // The residual of the next 64 columns is requested before the current
    // ones are stored (out may alias it, so the compiler cannot move a load
    // over a store: one by one they would cost a memory round trip each).
    constexpr bool kRes = EPI == FH_EPI_RESIDUAL;
    uint2 rv[kRes ? 2 : 1][kRes ? 16 : 1];
    auto load_residual = [&](auto slot_c, int p) {
      if constexpr (kRes) {
#pragma unroll
        for (int s = 0; s < 16; ++s) {
          const uint32_t row = min(row0 + 4 * s + (lane >> 4), m - 1);
          rv[decltype(slot_c)::value][s] =
              *reinterpret_cast<const uint2*>(residual + (uint64_t)row * ldo + bn * 16 + 64 * p + 4 * (lane & 15));
        }
      }
    };
    load_residual(std::integral_constant<int, 0>{}, 0);
    band_for<0, CG / 2>([&](auto p_c) {
      constexpr int p = decltype(p_c)::value;  // columns 64 p .. 64 p + 63 of the block
      if constexpr (p + 1 < CG / 2) load_residual(std::integral_constant<int, kRes ? (p + 1) % 2 : 0>{}, p + 1);
      if constexpr (p > 0) wave_fence();
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const f32x16& a = acc[2 * p + i][j];
            *reinterpret_cast<f32x4*>(stage + (32 * j + c) * kStagePitch + 32 * i + 8 * e + 4 * hi) =
                f32x4{a[4 * e], a[4 * e + 1], a[4 * e + 2], a[4 * e + 3]};
          }
      wave_fence();
      const uint32_t n0 = bn * 16 + 64 * p;
      if constexpr (EPI == FH_EPI_SWIGLU) {
        // Each 32 staged columns are a gate tile and its up tile. A wave
        // store covers 8 columns (two 4-column halves) of 32 rows: whole
        // 256-byte runs of the output's tile order.
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          const int g = s & 3, r = 32 * (s >> 2) + (lane >> 1), half = lane & 1;
          const int col = 32 * (g >> 1) + 8 * (g & 1) + 4 * half;
          const f32x4 gate = *reinterpret_cast<const f32x4*>(stage + r * kStagePitch + col);
          const f32x4 up = *reinterpret_cast<const f32x4*>(stage + r * kStagePitch + col + 16);
          if (row0 + r >= m) continue;
          uint32_t y[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = swiglu_bf16(round_bf16(gate[e]), round_bf16(up[e]), bad);
          *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out) +
                                    act_offset_m(row0 + r, n0 / 2 + 8 * g + 4 * half, mtiles)) =
              make_uint2(y[0] | (y[1] << 16), y[2] | (y[3] << 16));
        }
      } else {
#pragma unroll
        for (int s = 0; s < 16; ++s) {
          const int r = 4 * s + (lane >> 4), col = 4 * (lane & 15);
          const f32x4 v = *reinterpret_cast<const f32x4*>(stage + r * kStagePitch + col);
          if (row0 + r >= m) continue;
          const uint64_t o = (uint64_t)(row0 + r) * ldo + n0 + col;
          if constexpr (EPI == FH_EPI_F32) {
            *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(out) + o) = v;
          } else if constexpr (EPI == FH_EPI_BF16) {
            *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out) + o) =
                make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
          } else {
            const uint2 r0 = rv[p % 2][s];
            *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out) + o) =
                make_uint2(pack_bf16x2((0.0f + v[0]) + lo_bf16(r0.x), (0.0f + v[1]) + hi_bf16(r0.x)),
                           pack_bf16x2((0.0f + v[2]) + lo_bf16(r0.y), (0.0f + v[3]) + hi_bf16(r0.y)));
          }
        }
      }
    });
    if (bad) raise_error(err, ERR_NONFINITE);
  }
}

template <int EPI>
hipError_t launch_band(const uint16_t* xt, const uint16_t* w, uint32_t m, uint32_t n, uint32_t k,
                       const uint16_t* residual, void* out, uint32_t ldo, const QkvRopeArgs& qa, uint32_t* err,
                       hipStream_t s) {
  hipLaunchKernelGGL((gemm_band_kernel<EPI>), dim3(n / kBandCols, (m + kLargeBlockRows - 1) / kLargeBlockRows),
                     dim3(64 * kBandWaves), 0, s, xt, w, m, act_mtiles(m), k / 32, residual, out, ldo, qa, err);
  return hipGetLastError();
}

// (k < 2^24: a block's weight tiles are within the 32-bit offsets of its loads.)
bool band_ok(uint32_t m, uint32_t n, uint32_t k) {
  return m > kMaxRows && n % kBandCols == 0 && k % 32 == 0 && k > 0 && k < 1u << 24;
}

}  // namespace

// Estimated microseconds of a launch (fitted with mid_cost, k_gemm_mid.hip):
// rounds of the 256 CUs in units of a full block, at least one; a last block of
// at most 64 rows takes 0.59 of one, a longer one a quarter per 64 rows.
// Blocks that outnumber the CUs' rounds with less than their work leave some CU
// a full block and a last one: 600 x 12288 x 2048 SwiGLU is 288 blocks with the
// work of 240, 54 us (50 in 256 x 256 blocks), not the 37 of one round.
float gemm_band_cost(uint32_t m, uint32_t n, uint32_t k, uint32_t epilogue, bool fused_qkv) {
  if (!band_ok(m, n, k)) return -1.f;
  const uint32_t tail = m % kLargeBlockRows;
  const float part = tail == 0 ? 0.f : tail <= 64 ? 0.59f : (tail + 63) / 64 * 0.25f;
  const float bands = (float)(n / kBandCols);
  float rounds = ceilf(bands * (m / kLargeBlockRows + part) / 256.f);
  if (bands * ((m + kLargeBlockRows - 1) / kLargeBlockRows) > 256.f * rounds) rounds += part;
  const float around = fused_qkv                       ? 6.66f
                       : epilogue == FH_EPI_SWIGLU   ? 3.47f
                       : epilogue == FH_EPI_RESIDUAL ? 1.91f
                       : epilogue == FH_EPI_F32      ? 1.6f
                                                     : 1.79f;
  return 4.86f + rounds * (around + (k / 32) * 0.41f);
}

hipError_t launch_gemm_band(const uint16_t* x_tiled, const uint16_t* w_tiled, uint32_t m, uint32_t n, uint32_t k,
                            uint32_t epilogue, const uint16_t* residual, void* out, uint32_t ldo, uint32_t* err,
                            hipStream_t s) {
  if (!band_ok(m, n, k)) return hipErrorInvalidValue;
  const QkvRopeArgs none{};
  switch (epilogue) {
    case FH_EPI_BF16: return launch_band<FH_EPI_BF16>(x_tiled, w_tiled, m, n, k, residual, out, ldo, none, err, s);
    case FH_EPI_RESIDUAL: return launch_band<FH_EPI_RESIDUAL>(x_tiled, w_tiled, m, n, k, residual, out, ldo, none, err, s);
    case FH_EPI_SWIGLU: return launch_band<FH_EPI_SWIGLU>(x_tiled, w_tiled, m, n, k, residual, out, ldo, none, err, s);
    case FH_EPI_F32: return launch_band<FH_EPI_F32>(x_tiled, w_tiled, m, n, k, residual, out, ldo, none, err, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_gemm_band_qkv_rope(const uint16_t* x_tiled, const uint16_t* w_tiled, uint32_t m, uint32_t n,
                                     uint32_t k, const QkvRopeArgs& qa, hipStream_t s) {
  if (!band_ok(m, n, k) || n != (qa.qh + 2 * qa.kvh) * 128) return hipErrorInvalidValue;
  return launch_band<kBandEpiQkvRope>(x_tiled, w_tiled, m, n, k, nullptr, nullptr, 0u, qa, nullptr, s);
}

}  // namespace fh
