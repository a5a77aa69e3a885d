// K4 for prefill chunks of long runs of rows: causal attention of blocks of
// consecutive rows of one sequence. Same contract as k_attention_block.hip,
// which keeps the chunks of up to kPanelRows rows and those whose runs of rows
// are short (attention_prefill_form): for a row at position p, keys t = 0..p through the row's
// page table, score = (q . k_t) * f32(0x3db504f3), softmax, out = bf16(n / l)
// (device/qwen3-all-kernels-v1/src/paged_decode.rs:222-572).
//
// A workgroup owns one block (128 / G, 64 / G or 32 / G rows, by the form)
// and one KV head; a wave owns 32 query vectors (vector j: row j / G, head
// j % G), and the 4 waves share 64- or 128-key tiles of K and V, fetched global -> LDS directly (buffer
// loads, 16 bytes per lane, double-buffered). Slots past the block's last
// position are outside the loads' buffer bounds and arrive as zeros, so what
// an unwritten slot holds never meets an MFMA. Per tile and wave:
//   S^T = K Q^T on v_mfma_f32_32x32x16_bf16: lane l holds query l % 32 and,
//   of each 32 keys, keys 8 (e / 4) + 4 (l / 32) + e % 4 (e = 0..15), so the
//   softmax runs in the lane with one exchange between lanes l and l + 32;
//   online softmax per query on exp2 of (s - m) times the scale and log2 e in
//   one FMA. The running maximum m moves only when a tile's maximum exceeds
//   it by more than 8 in the exponent of 2 (terms then reach at most 2^8: no
//   precision is lost, and the 64 accumulators are rescaled rarely). Each
//   lane sums its own keys' terms; the two halves are added at the end;
//   O^T += V^T P^T on the same MFMA. P is FP32; it enters as two bf16 terms,
//   hi = bf16(p) and lo = bf16(p - hi) (within 2^-17 p of p), both products
//   accumulated in FP32. The B operand of keys 16 s .. 16 s + 15 is a lane's
//   own terms e = 8 (s % 2) .. + 7, which fixes the order of the 16 keys
//   inside the MFMA; the V^T operand follows it: two transposing LDS reads
//   (ds_read_b64_tr_b16: 16 lanes read 4 keys x 16 dims, each lane gets one
//   dim's 4 keys) of keys 16 s + 4 (l / 32) + 0..3 and the same + 8.
// LDS rows are 256 bytes (one token), their 16-byte chunks permuted so that
// the reads spread over the banks: K chunk c of key t at c ^ (t & 15), V
// chunk c at c ^ 4 (t & 3).
//
// What bounds it: 768 MFMA cycles per 32 queries x 32 keys (a third each for
// the scores and the two PV terms) against about as many VALU cycles (16
// exponentials, the split of P), two waves per SIMD: the matrix cores are 57 %
// busy at the 1.8 GHz the power limit leaves. us per layer, 16-row blocks with
// 16-key tiles (k_attention_block.hip) -> this kernel: one 8000-token 8B prompt
// 2010 -> 689, 32 prompts of 256 tokens 94 -> 63, one of 777 tokens 42 -> 22
// (29 without the waves along the keys), a 509-token 0.6B prompt 21 -> 13 (18).
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace fh {

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kPreWaves = 4;
// f32(0x3db504f3) (1/sqrt(128), paged_decode.rs:31-35) times log2 e.
constexpr float kScoreScale = 0.08838834764831845f;
constexpr float kLog2e = 1.44269504088896341f;

// WK: waves along the keys. WK = 1: 4 waves of 32 vectors (a block of 128),
// each taking every 32-key group of the 64-key tiles. WK = 2: 2 waves of
// vectors (64), two taking one key group each. WK = 4: 32 vectors, 128-key
// tiles, a key group per wave. The states of waves with the same vectors are
// merged through LDS at the end, in wave order.
template <int G, int WK>
__global__ __launch_bounds__(64 * kPreWaves, WK == 4 ? 1 : 2) void attn_prefill_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    const uint32_t* __restrict__ positions, const uint32_t* __restrict__ table, const uint32_t* __restrict__ blocks,
    uint16_t* __restrict__ out, uint32_t out_mtiles, uint32_t qh, uint32_t kvh, uint32_t stride, uint32_t pages,
    uint32_t context, uint32_t* err) {
  constexpr int WQ = kPreWaves / WK;             // waves along the vectors
  constexpr int kKeys = WK == 4 ? 128 : 64;      // keys per tile
  constexpr int kGroups = kKeys / 32 / WK;       // 32-key groups per wave and tile
  constexpr int kPages = kKeys / 16;             // pages per tile
  constexpr int kFetch = kPages / kPreWaves;     // of which each wave fetches this many
  constexpr size_t kTileBytes = sizeof(u32x4) * 2 * kKeys * 16;
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[2 * kTileBytes];
  auto& klds = *reinterpret_cast<u32x4(*)[2][kKeys][16]>(lds_raw);
  auto& vlds = *reinterpret_cast<u32x4(*)[2][kKeys][16]>(lds_raw + kTileBytes);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wq = wave / WK, wk = wave % WK;
  // KV heads vary fastest over the workgroups, which go to the 8 XCDs
  // round-robin: with 8 KV heads each XCD's L2 serves one head's K and V.
  const uint32_t h = blockIdx.x;
  auto uniform = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
  const uint32_t desc = uniform(blocks[blockIdx.y]);
  const uint32_t row0 = desc & 0xffffu, nrows = desc >> 16;
  const uint32_t last = row0 + nrows - 1;
  const uint32_t* trow = table + (uint64_t)last * stride;
  const uint32_t pos_last = uniform(positions[last]);
  const bool pos_ok = pos_last < context && pos_last / 16 < stride;
  if (!pos_ok && h == 0 && threadIdx.x == 0) raise_error(err, ERR_POSITION);
  const uint32_t pmax = pos_ok ? pos_last : 0u;
  const uint32_t npages = pmax / 16 + 1, tiles = pmax / kKeys + 1;

  // Page-table entries of 64 pages, one per lane, the next 64 requested ahead.
  auto table_chunk = [&](uint32_t first) { return first + lane < npages ? trow[first + lane] : 0u; };
  uint32_t tab = table_chunk(0), tab_next = table_chunk(64);

  // Wave w copies pages w, w + 4, ... of a tile, four tokens per load (lane:
  // token 4 i + lane / 16, LDS chunk lane % 16).
  const uint32_t token_bytes = kvh * 256;  // between consecutive tokens of one head
  uint32_t koff[4], voff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t row = (4 * i + (lane >> 4)) * token_bytes;
    koff[i] = row + (((lane & 15) ^ (4 * i + (lane >> 4))) & 15) * 16;
    voff[i] = row + (((lane & 15) ^ ((lane >> 4) << 2)) & 15) * 16;
  }
  uint32_t bad_page = 0;  // uniform
  auto fetch = [&](uint32_t t, int buf) {
#pragma unroll
    for (int f = 0; f < kFetch; ++f) {
      const uint32_t in_tile = wave + f * kPreWaves, pi = kPages * t + in_tile;
      uint32_t page = (uint32_t)__builtin_amdgcn_readlane((int)tab, (int)(pi & 63u));
      uint32_t valid = pi < npages ? min(16u, pmax + 1 - pi * 16) : 0u;  // written tokens of the page
      if (page >= pages) {
        bad_page |= valid;
        page = 0;
        valid = 0;
      }
      // Loads of tokens past the written ones are out of bounds and return zeros.
      const uint32_t bytes = valid * token_bytes;
      const uint64_t base = ((uint64_t)page * 16 * kvh + h) * 128;
      auto krs = __builtin_amdgcn_make_buffer_rsrc((void*)(kc + base), 0, bytes, 0x00020000);
      auto vrs = __builtin_amdgcn_make_buffer_rsrc((void*)(vc + base), 0, bytes, 0x00020000);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            krs, (__attribute__((address_space(3))) void*)&klds[buf][16 * in_tile + 4 * i][0], 16, koff[i], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            vrs, (__attribute__((address_space(3))) void*)&vlds[buf][16 * in_tile + 4 * i][0], 16, voff[i], 0, 0, 0);
    }
  };
  fetch(0, 0);

  // Query operand: lane l holds vector l % 32 of the wave, dims 16 i + 8 (l / 32) .. + 7.
  const uint32_t c = lane & 31, hi = lane >> 5;
  const uint32_t rj = (32 * wq + c) / G, head = h * G + c % G;
  const bool live = (uint32_t)(32 * wq / G) < nrows;  // a wave with no rows only fetches
  const bool qvalid = rj < nrows;
  // Vectors past the block's rows run with zero queries (and are not stored).
  const uint32_t qpos = qvalid ? positions[row0 + rj] : pmax;
  const uint32_t qpos_min = uniform(positions[row0 + min((uint32_t)(32 * wq / G), nrows - 1)]);  // of the wave's rows
  u32x4 qv[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    qv[i] = qvalid ? *reinterpret_cast<const u32x4*>(q + ((uint64_t)(row0 + rj) * qh + head) * 128 + 16 * i + 8 * hi)
                   : u32x4{0u, 0u, 0u, 0u};

  const float kNegInf = -__builtin_inff();
  const float cs = kScoreScale * kLog2e;
  float m_run = kNegInf, l_run = 0.f, s_abs = 0.f;
  f32x16 acc[4];  // output dims 32 d + 8 (e / 4) + 4 hi + e % 4 of vector c
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[d][e] = 0.f;

  // Lane parts of the LDS addresses.
  const u32x4* kl = &klds[0][c][0];
  const uint32_t kx = c & 15;
  // Transposing reads: lane j of 16 addresses key j / 4, dims 4 (j % 4) .. + 3.
  const uint32_t tj = lane & 15, tkey = 4 * hi + (tj >> 2);
  const uint32_t tchunk = ((lane >> 4) & 1) * 2 + ((tj & 3) >> 1), thalf = tj & 1;

  auto compute = [&](uint32_t t) {
    const int buf = t & 1;
    const int own = kGroups * wk;  // this wave's first 32-key group of the tile
    f32x16 s[kGroups];
#pragma unroll
    for (int kt = 0; kt < kGroups; ++kt) {
#pragma unroll
      for (int e = 0; e < 16; ++e) s[kt][e] = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const u32x4 ka = kl[(buf * kKeys + 32 * (own + kt)) * 16 + ((2 * i + hi) ^ kx)];
        s[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ka),
                                                        __builtin_bit_cast(bf16x8, qv[i]), s[kt], 0, 0, 0);
      }
    }
    const uint32_t first = t * kKeys + 32 * own, key0 = first + 4 * hi;
    if (first + 32 * kGroups - 1 > qpos_min) {
      // Keys past a row's position: no term (and no part in the finiteness check).
#pragma unroll
      for (int kt = 0; kt < kGroups; ++kt)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const bool ok = key0 + 32 * kt + 8 * (e >> 2) + (e & 3) <= qpos;
          s_abs = fmaxf(s_abs, ok ? __builtin_fabsf(s[kt][e]) : 0.f);
          s[kt][e] = ok ? s[kt][e] : kNegInf;
        }
    } else {
#pragma unroll
      for (int kt = 0; kt < kGroups; ++kt)
#pragma unroll
        for (int e = 0; e < 16; ++e) s_abs = fmaxf(s_abs, __builtin_fabsf(s[kt][e]));
    }
    float mt = kNegInf;
#pragma unroll
    for (int kt = 0; kt < kGroups; ++kt)
#pragma unroll
      for (int e = 0; e < 16; ++e) mt = fmaxf(mt, s[kt][e]);
    {
      // Lanes l and l + 32 hold the other half of the same query's keys.
      const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, mt), __builtin_bit_cast(uint32_t, mt),
                                                       false, false);
      mt = fmaxf(__builtin_bit_cast(float, (uint32_t)sw[0]), __builtin_bit_cast(float, (uint32_t)sw[1]));
    }
    // A wave along the keys may meet no key of a vector for some tiles (m_run
    // and mt both -inf: their difference is NaN, no move).
    if (__builtin_amdgcn_ballot_w64((mt - m_run) * cs > 8.f) != 0ull) {
      const float m_new = fmaxf(m_run, mt);
      const float alpha = m_run == kNegInf ? 0.f : __builtin_amdgcn_exp2f((m_run - m_new) * cs);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[d][e] *= alpha;
    }
    const float mc = WK > 1 && m_run == kNegInf ? 0.f : m_run * cs;
    float ps = 0.f;
#pragma unroll
    for (int g = 0; g < 2 * kGroups; ++g) {
      // Keys 16 g .. 16 g + 15 of the wave's groups.
      float p[8];
      uint32_t ph[4], pl[4];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[g >> 1][8 * (g & 1) + e], cs, -mc));
        ps += p[e];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        ph[e] = pack_bf16x2(p[2 * e], p[2 * e + 1]);
        pl[e] = pack_bf16x2(p[2 * e] - lo_bf16(ph[e]), p[2 * e + 1] - hi_bf16(ph[e]));
      }
      const bf16x8 bh = __builtin_bit_cast(bf16x8, u32x4{ph[0], ph[1], ph[2], ph[3]});
      const bf16x8 bl = __builtin_bit_cast(bf16x8, u32x4{pl[0], pl[1], pl[2], pl[3]});
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        u32x2 vq[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const uint32_t key = 32 * own + 16 * g + 8 * u + tkey;
          const uint32_t chunk = (4 * d + tchunk) ^ ((tj >> 2) << 2);
          auto* src = reinterpret_cast<u32x2*>(&vlds[buf][key][chunk]) + thalf;
          vq[u] = __builtin_bit_cast(
              u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)src));
        }
        const bf16x8 va = __builtin_bit_cast(bf16x8, u32x4{vq[0][0], vq[0][1], vq[1][0], vq[1][1]});
        acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, bh, acc[d], 0, 0, 0);
        acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, bl, acc[d], 0, 0, 0);
      }
    }
    l_run += ps;
  };
  for (uint32_t t = 0; t < tiles; ++t) {
    __builtin_amdgcn_s_waitcnt(0 | (7u << 4) | (15u << 8));  // this wave's share of tile t is in LDS
    __syncthreads();  // everyone's is, and everyone is done with tile t - 1
    if (t + 1 < tiles) {
      if ((t + 1) % (64 / kPages) == 0) {
        tab = tab_next;
        tab_next = table_chunk(kPages * (t + 1) + 64);
      }
      fetch(t + 1, (t + 1) & 1);
    }
    if (live) compute(t);
  }

  bool bad = false;
  float L = l_run;
  {
    const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, L), __builtin_bit_cast(uint32_t, L),
                                                     false, false);
    L = __builtin_bit_cast(float, (uint32_t)sw[0]) + __builtin_bit_cast(float, (uint32_t)sw[1]);
  }
  if constexpr (WK > 1) {
    // Waves wk > 0 hand their state over through the tiles' LDS: accumulators
    // as 16-byte words by lane, then m, l and the score bound of each lane.
    constexpr size_t kSlot = sizeof(f32x4) * 16 * 64 + sizeof(float) * 3 * 64;
    static_assert(kSlot * WQ * (WK - 1) <= sizeof(lds_raw), "one slot per wave handing over");
    auto slot_acc = [&](int k) { return reinterpret_cast<f32x4*>(lds_raw + kSlot * (wq * (WK - 1) + k - 1)); };
    __syncthreads();  // every wave is done with the tiles
    if (live && wk > 0) {
      f32x4* sa = slot_acc(wk);
      float* sm = reinterpret_cast<float*>(sa + 16 * 64);
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4)
          sa[(4 * d + e4) * 64 + lane] =
              f32x4{acc[d][4 * e4], acc[d][4 * e4 + 1], acc[d][4 * e4 + 2], acc[d][4 * e4 + 3]};
      sm[lane] = m_run;
      sm[64 + lane] = L;
      sm[128 + lane] = s_abs;
    }
    __syncthreads();
    if (live && wk == 0) {
#pragma unroll
      for (int k = 1; k < WK; ++k) {
        const f32x4* sa = slot_acc(k);
        const float* sm = reinterpret_cast<const float*>(sa + 16 * 64);
        const float mo = sm[lane], lo = sm[64 + lane];
        s_abs = fmaxf(s_abs, sm[128 + lane]);
        const float m_new = fmaxf(m_run, mo);
        const float fs = m_run == kNegInf ? 0.f : __builtin_amdgcn_exp2f((m_run - m_new) * cs);
        const float fo = mo == kNegInf ? 0.f : __builtin_amdgcn_exp2f((mo - m_new) * cs);
        m_run = m_new;
        L = L * fs + lo * fo;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[d][e] = acc[d][e] * fs + sa[(4 * d + (e >> 2)) * 64 + lane][e & 3] * fo;
      }
    }
  }
  if (live && wk == 0) {
    if (qvalid) {
      bad = !(L > 0.f) | !(s_abs < __builtin_inff());
      const float inv = __fdiv_rn(1.0f, L);
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
          const uint32_t w0 = pack_bf16x2(acc[d][4 * e4] * inv, acc[d][4 * e4 + 1] * inv);
          const uint32_t w1 = pack_bf16x2(acc[d][4 * e4 + 2] * inv, acc[d][4 * e4 + 3] * inv);
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            const uint32_t wd = b ? w1 : w0;
            bad |= ((wd & 0x7f80u) == 0x7f80u) | ((wd & 0x7f800000u) == 0x7f800000u);
          }
          const uint32_t col = head * 128 + 32 * d + 8 * e4 + 4 * hi;
          uint16_t* dst = out_mtiles ? out + act_offset_m(row0 + rj, col, out_mtiles)
                                     : out + (uint64_t)(row0 + rj) * qh * 128 + col;
          *reinterpret_cast<uint2*>(dst) = make_uint2(w0, w1);
        }
    }
  }
  if (bad) raise_error(err, ERR_NONFINITE);
  if (bad_page != 0 && lane == 0) raise_error(err, ERR_PAGE);
}

}  // namespace

namespace {

// What attention_prefill_form needs of each form: keys per tile (short blocks:
// four pages), workgroups that run at once (0: not a limit by itself), and
// microseconds per launch, per tile of one workgroup's chain, per workgroup and
// per tile of all of them (256 CUs), and per tile of each further round.
struct PrefillForm {
  uint32_t form, tile, slots;
  float launch_us, chain_us, group_us, tile_us, round_us;
};
constexpr PrefillForm kPrefillForms[] = {{0, 64, 0, 9.05f, 0.f, 0.f, 1.76f, 0.f},
                                         {1, 64, 512, 8.35f, 1.82f, 0.67f, 1.43f, 2.59f},
                                         {2, 64, 512, 8.24f, 1.24f, 1.91f, 0.87f, 1.62f},
                                         {4, 128, 256, 9.29f, 1.74f, 4.42f, 1.56f, 1.96f}};

}  // namespace

// The form with the lowest estimate: the longest workgroup's chain, the work
// of all of them, or rounds of average ones, whichever is longest. Its
// constants are fitted to the times of all forms over 1368 chunks of 257 to
// 8000 rows (1 to 2000 sequences of 1 to 5000 rows at contexts of 0 to 7000
// tokens, alone and mixed; 1, 2, 4 and 8 query heads per KV head): it picks a
// form 0.4 % slower than the fastest on average, 17 % at most (32 sequences of
// 24 rows on 3000 tokens, 84 us in short blocks, 99 taken), and never one more
// than 7 % slower than waves along the keys by the chunk's rows alone, as
// before. Those were 22 % slower than the fastest on average:
// a chunk of many short runs got long blocks that held a row or two. us per
// layer by the rows alone / now / short blocks: 0.6B 300 sequences of 1 row 67 /
// 14 / 14, 8B 300 x 1 68 / 17 / 17, 20 x 16 rows on 7000 tokens 288 / 198 / 191,
// 10 x 32 on 7000 241 / 181 / 187; 2 x 1000 rows 42 / 33 / 105.
uint32_t attention_prefill_form(const uint32_t* position, const uint32_t* rows, uint32_t nruns, uint32_t qh,
                                uint32_t kvh) {
  uint32_t best = 0;
  float best_us = 0.f;
  for (const PrefillForm& f : kPrefillForms) {
    const uint32_t bq = attention_prefill_block_rows(f.form, qh, kvh);
    uint64_t groups = 0, tiles = 0;
    uint32_t longest = 0;
    for (uint32_t i = 0; i < nruns; ++i)
      for (uint32_t r = 0; r < rows[i]; r += bq) {
        const uint32_t last = position[i] + (rows[i] - r < bq ? rows[i] : r + bq) - 1;
        const uint32_t t = last / f.tile + 1;
        ++groups;
        tiles += t;
        if (t > longest) longest = t;
      }
    const float n = (float)(groups * kvh), all = (float)(tiles * kvh), average = all / n;
    // Short blocks: 4, 2 or 1 page phases (launch_attention_blocks).
    const float chain = f.form ? f.chain_us : n <= 256.f ? 1.62f : n <= 512.f ? 2.81f : 3.69f;
    float us = fmaxf(chain * longest, (f.group_us * n + f.tile_us * all) / 256.f);
    if (f.slots) us = fmaxf(us, average * (chain + (ceilf(n / f.slots) - 1.f) * f.round_us));
    us += f.launch_us;
    if (f.form == 0 || us < best_us) {
      best = f.form;
      best_us = us;
    }
  }
  return best;
}

uint32_t attention_prefill_block_rows(uint32_t form, uint32_t qh, uint32_t kvh) {
  return form ? 128u / form / (qh / kvh) : attention_block_rows(qh, kvh);
}

hipError_t launch_attention_prefill(uint32_t form, const uint16_t* q, const uint16_t* k_cache,
                                    const uint16_t* v_cache, const uint32_t* positions, const uint32_t* table,
                                    const uint32_t* blocks, uint32_t nblocks, uint16_t* out, uint32_t out_tiled,
                                    uint32_t rows, uint32_t qh, uint32_t kvh, uint32_t stride, uint32_t pages,
                                    uint32_t context, uint32_t* err, hipStream_t s) {
  if (nblocks == 0) return hipSuccess;
  if (form != 1 && form != 2 && form != 4) return hipErrorInvalidValue;
  const uint32_t mt = out_tiled ? act_mtiles(rows) : 0u;
#define FH_PREFILL_WK(G_, WK_)                                                                            \
  hipLaunchKernelGGL((attn_prefill_kernel<G_, WK_>), dim3(kvh, nblocks), dim3(64 * kPreWaves), 0, s, q,   \
                     k_cache, v_cache, positions, table, blocks, out, mt, qh, kvh, stride, pages, context, err)
#define FH_PREFILL(G_)         \
  if (form == 1)               \
    FH_PREFILL_WK(G_, 1);      \
  else if (form == 2)          \
    FH_PREFILL_WK(G_, 2);      \
  else                         \
    FH_PREFILL_WK(G_, 4)
  switch (qh / kvh) {
    case 1: FH_PREFILL(1); break;
    case 2: FH_PREFILL(2); break;
    case 4: FH_PREFILL(4); break;
    case 8: FH_PREFILL(8); break;
    default: return hipErrorInvalidValue;
  }
#undef FH_PREFILL
#undef FH_PREFILL_WK
  return hipGetLastError();
}

}  // namespace fh
