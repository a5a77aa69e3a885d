// K1 projections of prefill chunks (m > 256 token rows) whose 256 x 256
// blocks fill the CUs, and the choice between this kernel and the ones with
// smaller blocks (k_gemm_band.hip, k_gemm_mid.hip): bf16 MFMA
// (v_mfma_f32_16x16x32_bf16), FP32 accumulation, compute-bound.
//
// Operands come from their tile orders (common.hpp): the weight in weight
// tile order and the activation in activation tile order with act_mtiles(m)
// row tiles, so every operand fetch of a wave is one contiguous 1 KiB in the
// exact MFMA register layout. A workgroup has 8 waves sharing each k-block's
// weight tiles through LDS; activation tiles are loaded by each wave. Each
// wave accumulates its MFMA tiles over the whole k range.
//
// Epilogues (same rounding points as the decode kernel, no split-K here):
//   FH_EPI_BF16     out[m][n] = bf16(acc)
//   FH_EPI_RESIDUAL out[m][n] = bf16((0 + acc) + residual[m][n]) (may alias out)
//   FH_EPI_SWIGLU   act = swiglu(bf16(gate), bf16(up)) in activation tile order
//                   (gate/up tiles interleaved by the weight layout)
//   FH_EPI_F32      out[m][n] = acc (FP32 logits)
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "../../include/ferric_hip.h"

namespace fh {

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));


__device__ __forceinline__ bf16x8 b8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

constexpr int kBigTiles = 16;  // 16-row tiles per block side (256 rows)

// 256 x 256 blocks for weights with n % 256 == 0 (every projection): 8 waves,
// each 8 n-tiles x 4 m-tiles (wave grid 2 along n x 4 along m). Only the
// weight tiles go through LDS: each k-block's 16 weight tiles are fetched
// global -> LDS directly (global_load_lds_dwordx4: lane i's 16 bytes land at
// tile + 16 i, the tile-order layout itself), 2 per wave, into an
// (LW + 1)-stage ring. Every wave loads its own 4 activation tiles straight
// into registers (an (LX + 1)-slot ring; a tile is used by the 2 waves along
// n, so it is fetched twice, the second time from the cache). Per k-block a
// workgroup reads
// 64 KiB out of LDS and writes 16 KiB; sharing the activation tiles through
// LDS as well (96 KiB read, 32 KiB written, the kernel this replaced) made
// LDS the bound, and this form is 14-28 % faster on the 8B projections with
// bit-identical results. Barriers are bare s_barrier: __syncthreads()' fence
// would wait for every load in flight, k-blocks ahead included.
//
// Counters on the gate/up projection (8192 x 24576 x 4096): 100.7M MFMAs of
// 16 cycles keep the MFMA pipe busy 66 % of the kernel's cycles (down 69 %,
// O 58 %, fused QKV 56 %) with no LDS bank conflicts; the library GEMM
// reaches 85 % on the gate/up shape but at a lower clock under the board's
// power limit, about 10 % faster in time.
constexpr unsigned xd_wait_vm(unsigned n) { return (n & 15u) | ((n >> 4) << 14) | (7u << 4) | (15u << 8); }

// Calls f(std::integral_constant<int, I>) for I = B .. E - 1, unrolled at compile time.
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// LX / LW: how many k-blocks ahead the activation / weight tiles are
// requested (LW >= LX, so W(kb) is always older than X(kb)). Measured on the
// 8B projections at m = 8192: LX = 3, LW = 4 is 2-7 % faster than 2 / 3
// (212 VGPRs, 80 KiB LDS, still 2 waves per SIMD); deeper rings, reading all
// of a k-block's weight tiles out of LDS up front, and two k-blocks per
// barrier were not faster.
//
// EPI == kEpiQkvRope (the QKV projection of a prefill chunk): a wave's 8
// n-tiles are exactly one head (128 columns) of 64 rows. After the k loop the
// wave stages them in LDS as bf16 rows (the projection's rounding) and runs
// their QK-norm, RoPE and KV append (qknorm_rope_kv_wave, qk_head.hpp): the
// same code and order as the kernel of many rows, without the QKV output's
// round trip through HBM or a second launch.
constexpr int kEpiQkvRope = 16;

template <int EPI, int LX = 3, int LW = 4>
__global__ __launch_bounds__(512) void gemm_large_xd_kernel(const uint16_t* __restrict__ xt,
                                                            const uint16_t* __restrict__ w, uint32_t m,
                                                            uint32_t mtiles, uint32_t kb_count,
                                                            const uint16_t* residual, void* out, uint32_t ldo,
                                                            uint32_t out_mtiles, const QkvRopeArgs qa,
                                                            uint32_t* err) {
  static_assert(LX >= 1 && LW >= LX, "weights requested no later than activations");
  constexpr int WN = 8, WM = 4, WSTAGES = LW + 1, XSLOTS = LX + 1;
  // The wait before k-block kb counts per kind: direct-to-LDS loads (the
  // weight tiles) and register loads (the activation tiles) complete out of
  // order with respect to each other, only loads of one kind in issue order.
  // If W(kb) were outstanding, so would be the 2 (LW - 1) weight loads after
  // it; if X(kb) were, the WM (LX - 1) activation loads after it. At most the
  // smaller count outstanding covers both.
  constexpr unsigned kWLater = 2 * (LW - 1), kXLater = WM * (LX - 1);
  constexpr unsigned kInFlight = kWLater < kXLater ? kWLater : kXLater;
  static_assert(kInFlight < 64, "vmcnt range");
  constexpr size_t kRingBytes = sizeof(u32x4) * WSTAGES * kBigTiles * 64;
  constexpr size_t kStageBytes = EPI == kEpiQkvRope ? 4ull * 8 * 64 * kQkPitch : 0;
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[kRingBytes > kStageBytes ? kRingBytes : kStageBytes];
  auto& wlds = *reinterpret_cast<u32x4(*)[WSTAGES][kBigTiles][64]>(lds_raw);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Block order by XCD: workgroups go to the 8 XCDs round-robin in dispatch
  // order, so with the plain order each XCD's co-resident workgroups cover
  // 12 n-blocks x 3 m-blocks (8B gate/up) and its L2 holds that many weight
  // and activation k-slices. Here XCD j takes m-blocks j, j + 8, ... four at
  // a time and walks all n-blocks with them: its workgroups cover 4 m x 8 n
  // blocks, fewer distinct operands per k-block (gate/up -4 %, O -8 %, QKV
  // and down unchanged at 8192 rows; outputs identical). Grids whose m-block
  // count is not a multiple of 32 keep the plain order.
  uint32_t gx = blockIdx.x, gy = blockIdx.y;
  if (gridDim.y % 32 == 0) {
    const uint32_t NB = gridDim.x, b = blockIdx.x + NB * blockIdx.y;
    const uint32_t r = b >> 3;  // position within this XCD's share
    const uint32_t group = r / (4 * NB), within = r % (4 * NB);
    gy = (group * 4 + within % 4) * 8 + (b & 7u);
    gx = within / 4;
  }
  const uint32_t bn = gx * kBigTiles, bm = gy * kBigTiles;
  const int wn = wave % 2, wm = wave / 2;
  const uint32_t last = kb_count - 1;
  // The fused QKV epilogue's row lookups (position, page, slot) are
  // requested now and used after the k loop.
  QkvRowSlot row_slot{0u, 0u, false};
  if constexpr (EPI == kEpiQkvRope) {
    const uint32_t row = (bm + wm * 4) * 16 + lane;
    if (row < m) row_slot = qkv_row_slot(row, qa);
  }
  // Weight fetch: tiles 2 wave, 2 wave + 1 of the block.
  const u32x4* wsrc = reinterpret_cast<const u32x4*>(w) + (uint64_t)(bn + 2 * wave) * kb_count * 64 + lane;
  const uint64_t w_tile = (uint64_t)kb_count * 64;
  auto fetch_w = [&](uint32_t kb) {
    const uint32_t k = min(kb, last);
#pragma unroll
    for (int t = 0; t < 2; ++t)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(wsrc + t * w_tile + (uint64_t)k * 64),
                                       (__attribute__((address_space(3))) void*)&wlds[kb % WSTAGES][2 * wave + t][0],
                                       16, 0, 0);
  };
  // Activation tiles of this wave: (kb, bm + wm * WM + j), into register slot S.
  const u32x4* xsrc = reinterpret_cast<const u32x4*>(xt) + (uint64_t)(bm + wm * WM) * 64 + lane;
  const uint64_t x_kb = (uint64_t)mtiles * 64;
  u32x4 xr[XSLOTS][WM];
  auto load_x = [&](auto slot_c, uint32_t kb) {
    const uint64_t k = min(kb, last);
#pragma unroll
    for (int j = 0; j < WM; ++j) xr[decltype(slot_c)::value][j] = xsrc[k * x_kb + j * 64];
  };

  f32x4 acc[WN][WM];
#pragma unroll
  for (int i = 0; i < WN; ++i)
#pragma unroll
    for (int j = 0; j < WM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Issue order per iteration j: W(j + LW), then X(j + LX); k-blocks past
  // the end are clamped to the last one, so the count of loads in flight is
  // the same at every iteration. The prologue issues in that same order (for
  // LX = 3, LW = 4: W0 W1 X0 W2 X1 W3 X2), so the first iteration's wait
  // covers X0 as well. Issued in another order the compiler adds its own wait for X0
  // inside the loop, and with direct-to-LDS loads in flight that wait is
  // vmcnt(0), draining every load once per loop iteration.
  static_for<0, LW>([&](auto j_c) {
    constexpr int j = decltype(j_c)::value - LW;
    fetch_w(j + LW);
    if constexpr (j + LX >= 0) load_x(std::integral_constant<int, (j + LX) % XSLOTS>{}, j + LX);
  });
  auto step = [&](auto s_c, uint32_t kb) {
    constexpr int S = decltype(s_c)::value;
    __builtin_amdgcn_s_waitcnt(xd_wait_vm(kInFlight));
    __builtin_amdgcn_s_barrier();  // W(kb) of every wave is in LDS
    fetch_w(kb + LW);
    load_x(std::integral_constant<int, (S + LX) % XSLOTS>{}, kb + LX);
    const int st = kb % WSTAGES;
#pragma unroll
    for (int i = 0; i < WN; ++i) {
      const u32x4 wv = wlds[st][wn * WN + i][lane];
#pragma unroll
      for (int j = 0; j < WM; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b8(wv), b8(xr[S][j]), acc[i][j], 0, 0, 0);
    }
  };
  uint32_t kb = 0;
  for (; kb + XSLOTS <= kb_count; kb += XSLOTS)
    static_for<0, XSLOTS>([&](auto s_c) { step(s_c, kb + decltype(s_c)::value); });
  static_for<0, XSLOTS - 1>([&](auto s_c) {
    if (kb + decltype(s_c)::value < kb_count) step(s_c, kb + decltype(s_c)::value);
  });
  __builtin_amdgcn_s_waitcnt(xd_wait_vm(0));

  const uint32_t nt0 = bn + wn * WN, mt0 = bm + wm * WM;
  const uint32_t q = lane >> 4, c = lane & 15;
  if constexpr (EPI == kEpiQkvRope) {
    __syncthreads();  // every wave is done reading the weight ring, which the staging reuses
    if (mt0 * 16 >= m) return;  // this wave's rows are all padding
    // D layout: lane l, element e holds column 16 i + 4 (l / 16) + e of the
    // head and row 16 j + l % 16 of the wave's 64 rows.
    uint32_t* rows_lds = reinterpret_cast<uint32_t*>(lds_raw) + (uint32_t)wave * 64 * kQkPitch;
#pragma unroll
    for (int j = 0; j < WM; ++j)
#pragma unroll
      for (int i = 0; i < WN; ++i) {
        const uint2 v = make_uint2(f32_to_bf16(acc[i][j][0]) | (f32_to_bf16(acc[i][j][1]) << 16),
                                   f32_to_bf16(acc[i][j][2]) | (f32_to_bf16(acc[i][j][3]) << 16));
        *reinterpret_cast<uint2*>(rows_lds + (16 * j + c) * kQkPitch + 8 * i + 2 * q) = v;
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    qknorm_rope_kv_wave<64>(rows_lds, mt0 * 16, m, gx * 2 + wn, qa, row_slot);
    return;
  }
  if (mt0 * 16 >= m) return;  // this wave's rows are all padding
  if constexpr (EPI == FH_EPI_SWIGLU) {
    bool bad = false;
#pragma unroll
    for (int p = 0; p < WN / 2; ++p) {
      const uint32_t col = ((nt0 + 2 * p) / 2) * 16 + 4 * q;
#pragma unroll
      for (int j = 0; j < WM; ++j) {
        const uint32_t row = (mt0 + j) * 16 + c;
        if (row >= m) continue;
        uint32_t y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          y[e] = swiglu_bf16(round_bf16(acc[2 * p][j][e]), round_bf16(acc[2 * p + 1][j][e]), bad);
        uint2 v = make_uint2(y[0] | (y[1] << 16), y[2] | (y[3] << 16));
        *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out) + act_offset_m(row, col, out_mtiles)) = v;
      }
    }
    if (bad) raise_error(err, ERR_NONFINITE);
  } else {
#pragma unroll
    for (int i = 0; i < WN; ++i) {
      const uint32_t n = (nt0 + i) * 16 + 4 * q;
#pragma unroll
      for (int j = 0; j < WM; ++j) {
        const uint32_t row = (mt0 + j) * 16 + c;
        if (row >= m) continue;
        const uint64_t o = (uint64_t)row * ldo + n;
        if constexpr (EPI == FH_EPI_F32) {
          *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(out) + o) = acc[i][j];
        } else if constexpr (EPI == FH_EPI_BF16) {
          uint2 v = make_uint2(f32_to_bf16(acc[i][j][0]) | (f32_to_bf16(acc[i][j][1]) << 16),
                               f32_to_bf16(acc[i][j][2]) | (f32_to_bf16(acc[i][j][3]) << 16));
          *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out) + o) = v;
        } else {
          const uint2 rv = *reinterpret_cast<const uint2*>(residual + o);
          const float r0 = lo_bf16(rv.x), r1 = hi_bf16(rv.x), r2 = lo_bf16(rv.y), r3 = hi_bf16(rv.y);
          uint2 v = make_uint2(f32_to_bf16((0.0f + acc[i][j][0]) + r0) | (f32_to_bf16((0.0f + acc[i][j][1]) + r1) << 16),
                               f32_to_bf16((0.0f + acc[i][j][2]) + r2) | (f32_to_bf16((0.0f + acc[i][j][3]) + r3) << 16));
          *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out) + o) = v;
        }
      }
    }
  }
}

// Estimated microseconds of a launch of 256 x 256 blocks (fitted with
// mid_cost, k_gemm_mid.hip): whole rounds of the 256 CUs, a k-block taking
// longer the more CUs run, and what a block costs around its k loop.
float block_cost(uint32_t m, uint32_t n, uint32_t k, uint32_t epilogue, bool fused_qkv) {
  const uint32_t blocks = n / (16 * kBigTiles) * ((m + 255) / 256);
  const float kb_us = blocks < 100 ? 0.477f : blocks < 256 ? 0.607f : 0.688f;
  const float around =
      fused_qkv ? 11.86f : epilogue == FH_EPI_SWIGLU ? 10.83f : epilogue == FH_EPI_RESIDUAL ? 25.58f : 15.26f;
  return ((blocks + 255) / 256) * (around + (k / 32) * kb_us);
}

// Which of the three kernels a projection of m rows runs.
enum class LargeKernel { kMid, kBand, kBlock };

LargeKernel pick_kernel(uint32_t m, uint32_t n, uint32_t k, uint32_t epilogue, bool fused_qkv) {
  const float mid = gemm_mid_cost(m, n, k, epilogue, fused_qkv), band = gemm_band_cost(m, n, k, epilogue, fused_qkv);
  const bool block_ok = m > kPanelRows && n % (16 * kBigTiles) == 0;
  const float block = block_ok ? block_cost(m, n, k, epilogue, fused_qkv) : -1.f;
  if (block_ok && block <= mid && (band < 0.f || block <= band)) return LargeKernel::kBlock;
  return band >= 0.f && band < mid ? LargeKernel::kBand : LargeKernel::kMid;
}

// Whether a SwiGLU or FP32 projection of up to kPanelRows rows streams its
// weight through the panel kernel: where its 128-column slices fill more than
// half of the CUs, up to 224 rows. Fewer slices leave too many CUs idle, and
// with more rows the panel's LDS traffic exceeds its weight stream. Panel
// against the fastest block (us, cold weights): 152 slices (19456 x 2560) 64 rows
// 25 / 27, 160 rows 36 / 39; 128 slices (16384 x 4096) 40 rows 33 / 29, 160 rows
// 48 / 43; 48 slices (6144 x 1024) 48 rows 10.8 / 6.5, 160 rows 17.6 / 9.5; 32
// slices (4096 x 4096) 30 / 12.5, 44 / 18.7; 192 slices (24576 x 4096) 64 rows
// 37 / 42, 160 rows 53 / 63, 224 rows 69 / 71, 240 rows 75 / 69; 1187 slices
// (151936 x 4096) 64 rows 230 / 250, 160 rows 284 / 313, 240 rows 400 / 357. The
// line is not the faster side everywhere: the panel's time steps at 97 and 161
// rows (gate/up at 100 to 128 rows 56 / 53, the head of 4096 at 192 to 224 rows
// 334 / 315 to 384 / 356), and a head of 1024 columns is up to 9 % faster in
// blocks below 65 rows (48 rows 70 / 66) and up to 21 % above 160 (208 rows 131 /
// 108). Both sides ran the panel before the blocks.
bool panel_streams(uint32_t m, uint32_t n) { return m <= 224 && n > 128 * kPanelCols; }

}  // namespace

uint32_t gemm_block(uint32_t m, uint32_t n, uint32_t k, uint32_t epilogue, bool fused_qkv) {
  if (m <= kMaxRows || n == 0 || n % kPanelCols != 0 || k == 0 || k % 32 != 0) return 0;
  if (fused_qkv) {
    if (m <= kPanelRows || n % (16 * kBigTiles) != 0) return 0;
  } else if (epilogue > FH_EPI_F32 ||
             ((epilogue == FH_EPI_SWIGLU || epilogue == FH_EPI_F32) && panel_streams(m, n))) {
    return 0;
  }
  switch (pick_kernel(m, n, k, epilogue, fused_qkv)) {
    case LargeKernel::kMid: return gemm_mid_block(m, n, k, epilogue, fused_qkv);
    case LargeKernel::kBand: return kLargeBlockRows << 16 | kPanelCols;
    case LargeKernel::kBlock: break;
  }
  return (16 * kBigTiles) << 16 | 16 * kBigTiles;
}

hipError_t launch_gemm_qkv_rope(const uint16_t* x_tiled, const uint16_t* w_tiled, uint32_t m, uint32_t n, uint32_t k,
                                const QkvRopeArgs& qa, hipStream_t s) {
  const uint32_t mtiles = act_mtiles(m);
  if (m <= kPanelRows || n % (16 * kBigTiles) != 0 || k % 32 != 0 || mtiles % kBigTiles != 0 ||
      n != (qa.qh + 2 * qa.kvh) * 128)
    return hipErrorInvalidValue;
  switch (pick_kernel(m, n, k, FH_EPI_BF16, true)) {
    case LargeKernel::kMid: return launch_gemm_mid_qkv_rope(x_tiled, w_tiled, m, n, k, qa, s);
    case LargeKernel::kBand: return launch_gemm_band_qkv_rope(x_tiled, w_tiled, m, n, k, qa, s);
    case LargeKernel::kBlock: break;
  }
  const dim3 grid(n / (16 * kBigTiles), mtiles / kBigTiles);
  hipLaunchKernelGGL((gemm_large_xd_kernel<kEpiQkvRope>), grid, dim3(512), 0, s, x_tiled, w_tiled, m, mtiles, k / 32,
                     (const uint16_t*)nullptr, (void*)nullptr, 0u, 0u, qa, (uint32_t*)nullptr);
  return hipGetLastError();
}

hipError_t launch_gemm_large(const uint16_t* x_tiled, const uint16_t* w_tiled, uint32_t m, uint32_t n, uint32_t k,
                             uint32_t epilogue, const uint16_t* residual, void* out, uint32_t ldo, uint32_t* err,
                             hipStream_t s) {
  if (m <= kMaxRows) return launch_gemm(x_tiled, w_tiled, m, n, k, epilogue, 1, residual, out, ldo, err, s);
  if (n % kPanelCols != 0 || k % 32 != 0) return hipErrorInvalidValue;
  if ((epilogue == FH_EPI_SWIGLU || epilogue == FH_EPI_F32) && panel_streams(m, n))
    return launch_gemm(x_tiled, w_tiled, m, n, k, epilogue, 1, residual, out, ldo, err, s);
  switch (pick_kernel(m, n, k, epilogue, false)) {
    case LargeKernel::kMid:
      return launch_gemm_mid(x_tiled, w_tiled, m, n, k, epilogue, residual, out, ldo, err, s);
    case LargeKernel::kBand:
      return launch_gemm_band(x_tiled, w_tiled, m, n, k, epilogue, residual, out, ldo, err, s);
    case LargeKernel::kBlock: break;
  }
  const uint32_t mtiles = act_mtiles(m), kb = k / 32;
  const uint32_t out_mtiles = epilogue == FH_EPI_SWIGLU ? mtiles : 0u;
  const dim3 grid(n / (16 * kBigTiles), mtiles / kBigTiles);
#define FH_BIG(E)                                                                                           \
  hipLaunchKernelGGL((gemm_large_xd_kernel<E>), grid, dim3(512), 0, s, x_tiled, w_tiled, m, mtiles, kb, residual, \
                     out, ldo, out_mtiles, QkvRopeArgs{}, err)
  switch (epilogue) {
    case FH_EPI_BF16: FH_BIG(FH_EPI_BF16); break;
    case FH_EPI_RESIDUAL: FH_BIG(FH_EPI_RESIDUAL); break;
    case FH_EPI_SWIGLU: FH_BIG(FH_EPI_SWIGLU); break;
    case FH_EPI_F32: FH_BIG(FH_EPI_F32); break;
    default: return hipErrorInvalidValue;
  }
#undef FH_BIG
  return hipGetLastError();
}

}  // namespace fh
