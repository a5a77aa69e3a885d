// QK-norm + RoPE + paged KV append of bf16 QKV rows staged in LDS (the prefill
// path: the fused epilogues of the QKV projection kernels and the kernel of
// many rows), and its parts.
//
// Reference semantics: qwen3_rmsnorm_v1 at width 128 per head
// (device/qwen3-all-kernels-v1/src/rmsnorm.rs:380-526; the serial sum of
// squares of rmsnorm.rs:421-438, each square rounded before the add),
// qwen3_rope_v1 (rope_kv.rs:102: a' = a c - b s, b' = b c + a s on pairs
// (i, i + 64)), and qwen3_paged_kv_write_v1 (rope_kv.rs:261-388: K rotated,
// V raw, slot pages[pos / 16] * 16 + pos % 16).
#pragma once

#include "common.hpp"

namespace fh {

typedef unsigned int qk_u32x4 __attribute__((ext_vector_type(4)));

// Correctly rounded square root of a positive normal float. The hardware
// square root (v_sqrt_f32, what __fsqrt_rn becomes on this target) is only
// within 1 ulp, so one correction step picks among its estimate s and the
// neighbours s- and s+: the root rounds down to s- exactly when
// x <= s- * s, and up to s+ exactly when x > s+ * s (both products exact
// inside the FMA). A float x and either product differ by a multiple of
// ulp(s)^2, while these thresholds sit within ulp(s)^2 / 4 of the true
// rounding midpoints, so the comparisons decide exactly as the midpoints
// would. Below 2^-64 those differences would underflow, so x is first
// scaled by 2^64 and the root by 2^-32 (both exact). Checked against the
// midpoint definition for every positive normal float.
__device__ __forceinline__ float sqrt_rn(float x) {
  const bool tiny = x < 0x1p-64f;
  const float xs = tiny ? x * 0x1p64f : x;
  const float s = __builtin_amdgcn_sqrtf(xs);
  const uint32_t u = __builtin_bit_cast(uint32_t, s);
  const float down = __builtin_bit_cast(float, u - 1u), up = __builtin_bit_cast(float, u + 1u);
  float r = s;
  if (__builtin_fmaf(-down, s, xs) <= 0.0f) r = down;
  if (__builtin_fmaf(-up, s, xs) > 0.0f) r = up;
  return tiny ? r * 0x1p-32f : r;
}

// Inverse RMS exactly as qwen3_rmsnorm_v1 forms it
// (device/qwen3-all-kernels-v1/src/rmsnorm.rs:440-456): mean = sum / width
// (a division), + epsilon, correctly rounded sqrt, then 1 / sqrt.
__device__ __forceinline__ float inverse_rms(float sum, float width, float eps) {
  float mean_square = __fdiv_rn(sum, width);
  float stabilized = mean_square + eps;
  float denominator = sqrt_rn(stabilized);
  return __fdiv_rn(1.0f, denominator);
}

// Normalize-then-round, weight, round again (rmsnorm.rs:486-503; the witness
// in device/qwen3-rmsnorm-v1/tests/reference.rs:264-274 pins the double round).
__device__ __forceinline__ uint32_t norm_weight_bf16(float x, float inv, float w) {
  float normalized = round_bf16(x * inv);
  return f32_to_bf16(normalized * w);
}

// QK-norm + RoPE of one normalized head held by a wave: lane l holds
// elements l (a) and l + 64 (b) as bf16-valued floats, wa/wb the norm
// weights of those elements, c/s the RoPE factors of pair l at the row's
// position. The square sum runs serially in element order 0..127 (one
// rounding per square and per add, rmsnorm.rs:421-438) through lane reads.
// ra/rb: the rotated bf16 outputs of elements l and l + 64. Returns true
// when a value or the sum is nonfinite. The decode QK-norm kernel and the
// decode attention kernel's fused form both call this, so their outputs are
// bit-identical.
// The part after the square sum, given it (the block attention forms the
// sums of its heads another way, in the same order).
__device__ __forceinline__ bool qknorm_rope_wave_head_from_sum(float a, float b, float sum, float wa, float wb,
                                                               float c, float s, float eps, uint32_t& ra,
                                                               uint32_t& rb) {
  bool bad = !is_finite_f32(a) | !is_finite_f32(b);
  const float inv = inverse_rms(sum, 128.0f, eps);
  bad |= !is_finite_f32(sum) | !is_finite_f32(inv);
  const float an = bf16_to_f32(norm_weight_bf16(a, inv, wa));
  const float bn = bf16_to_f32(norm_weight_bf16(b, inv, wb));
  const float a_cos = an * c, b_sin = bn * s, b_cos = bn * c, a_sin = an * s;
  ra = f32_to_bf16(a_cos - b_sin);
  rb = f32_to_bf16(b_cos + a_sin);
  bad |= ((ra & 0x7f80u) == 0x7f80u) | ((rb & 0x7f80u) == 0x7f80u);
  return bad;
}

__device__ __forceinline__ bool qknorm_rope_wave_head(float a, float b, float wa, float wb, float c, float s,
                                                      float eps, uint32_t& ra, uint32_t& rb) {
  const float sqa = a * a, sqb = b * b;
  float sum = 0.f;
#pragma unroll
  for (int l = 0; l < 64; ++l) sum = sum + lane_bcast(sqa, l);
#pragma unroll
  for (int l = 0; l < 64; ++l) sum = sum + lane_bcast(sqb, l);
  return qknorm_rope_wave_head_from_sum(a, b, sum, wa, wb, c, s, eps, ra, rb);
}

struct QkvRopeArgs {
  const uint16_t* q_norm;
  const uint16_t* k_norm;
  const float* cos_t;  // [context][64]
  const float* sin_t;
  const uint32_t* positions;
  const uint32_t* table;  // [rows][stride]
  uint16_t* q_out;        // [rows][qh][128]
  uint16_t* k_cache;      // [pages][16][kvh][128]
  uint16_t* v_cache;
  uint32_t qh, kvh, stride, pages, context;
  float eps;
  uint32_t* err;
};

// A row's position and KV slot (slot_ok false: position or page outside the
// envelope; nothing is written to the cache then, and head 0 reports it).
struct QkvRowSlot {
  uint32_t pos, slot;
  bool slot_ok;
};

__device__ __forceinline__ QkvRowSlot qkv_row_slot(uint32_t row, const QkvRopeArgs& a) {
  QkvRowSlot r{a.positions[row], 0u, false};
  r.slot_ok = r.pos < a.context && r.pos / 16 < a.stride;
  if (r.slot_ok) {
    const uint32_t page = a.table[(uint64_t)row * a.stride + r.pos / 16];
    r.slot_ok = page < a.pages;
    r.slot = (page * 16u + (r.pos & 15u)) * a.kvh;
  }
  return r;
}

// Words per staged head row in LDS: 64 (128 bf16) + 4, so that rows stay
// 16-byte aligned and the lanes' row reads spread over the banks.
constexpr uint32_t kQkPitch = 68;

// The sum of a staged head's 128 squares in element order, each square
// rounded before the add: the only serial part.
__device__ __forceinline__ float qk_square_sum(const uint32_t* x) {
  const qk_u32x4* xr = reinterpret_cast<const qk_u32x4*>(x);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const qk_u32x4 v = xr[i];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float e0 = lo_bf16(v[k]), e1 = hi_bf16(v[k]);
      const float s0 = e0 * e0, s1 = e1 * e1;
      sum = sum + s0;
      sum = sum + s1;
    }
  }
  return sum;
}

// Dims 8 g .. 8 g + 7 and the same + 64 of a staged head x: normalized with
// inv and rotated (query heads 0 .. qh - 1, to q_out; key heads qh ..
// qh + kvh - 1, to the row's KV slot) or copied (value heads, to the slot).
// Returns whether an output is nonfinite (value heads are not checked).
__device__ __forceinline__ bool qknorm_rope_kv_piece(const uint32_t* x, uint32_t g, float inv, uint32_t row,
                                                     uint32_t head, const QkvRopeArgs& a, const QkvRowSlot rs) {
  const uint32_t heads = a.qh + a.kvh;
  qk_u32x4 xa = *reinterpret_cast<const qk_u32x4*>(x + 4 * g), xb = *reinterpret_cast<const qk_u32x4*>(x + 32 + 4 * g);
  uint16_t* dst = nullptr;
  bool bad = false;
  if (head >= heads) {
    if (rs.slot_ok) dst = a.v_cache + ((uint64_t)rs.slot + (head - heads)) * 128;
  } else {
    if (head < a.qh)
      dst = a.q_out + ((uint64_t)row * a.qh + head) * 128;
    else if (rs.slot_ok)
      dst = a.k_cache + ((uint64_t)rs.slot + (head - a.qh)) * 128;
    const uint16_t* wn = head < a.qh ? a.q_norm : a.k_norm;
    const qk_u32x4 wa = *reinterpret_cast<const qk_u32x4*>(wn + 8 * g);
    const qk_u32x4 wb = *reinterpret_cast<const qk_u32x4*>(wn + 64 + 8 * g);
    const uint64_t trig = (uint64_t)(rs.pos < a.context ? rs.pos : 0) * 64 + 8 * g;
    const float4* ct = reinterpret_cast<const float4*>(a.cos_t + trig);
    const float4* st = reinterpret_cast<const float4*>(a.sin_t + trig);
    const float4 c0 = ct[0], c1 = ct[1], s0 = st[0], s1 = st[1];
    const float cs[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
    const float sn[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      uint32_t oa[2], ob[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float an = bf16_to_f32(norm_weight_bf16(e ? hi_bf16(xa[k]) : lo_bf16(xa[k]), inv,
                                                      e ? hi_bf16(wa[k]) : lo_bf16(wa[k])));
        const float bn = bf16_to_f32(norm_weight_bf16(e ? hi_bf16(xb[k]) : lo_bf16(xb[k]), inv,
                                                      e ? hi_bf16(wb[k]) : lo_bf16(wb[k])));
        const float c = cs[2 * k + e], s = sn[2 * k + e];
        const float a_cos = an * c, b_sin = bn * s, b_cos = bn * c, a_sin = an * s;
        oa[e] = f32_to_bf16(a_cos - b_sin);
        ob[e] = f32_to_bf16(b_cos + a_sin);
        bad |= ((oa[e] & 0x7f80u) == 0x7f80u) | ((ob[e] & 0x7f80u) == 0x7f80u);
      }
      xa[k] = oa[0] | (oa[1] << 16);
      xb[k] = ob[0] | (ob[1] << 16);
    }
  }
  if (dst) {
    *reinterpret_cast<qk_u32x4*>(dst + 8 * g) = xa;
    *reinterpret_cast<qk_u32x4*>(dst + 64 + 8 * g) = xb;
  }
  return bad;
}

// kRows (16, 32 or 64) consecutive rows of one head, staged in LDS by this
// wave (or behind a barrier): lane l < kRows adds row l's squares, then 8
// lanes per row normalize, rotate and store whole 16-byte pieces, 8 rows at a
// time. rs: lane l's row row0 + l. One lane per row for everything stored 256
// bytes per lane and, in the kernels whose waves share a head's rows, left
// half of the waves or more idle. us per launch of the fused projection with
// one lane per row / this: 8000 rows of the 8B 372 / 333 (256 x 256 blocks),
// 777 rows 64.6 / 60.5 (256 x 128), 0.6B 1200 rows 26.9 / 22.0, 509 rows 18.1
// / 13.6 (128 x 64); bit-identical.
template <int kRows>
__device__ __forceinline__ void qknorm_rope_kv_wave(const uint32_t* staged, uint32_t row0, uint32_t m, uint32_t head,
                                                    const QkvRopeArgs& a, const QkvRowSlot rs) {
  const uint32_t lane = threadIdx.x & 63u, count = row0 < m ? min(m - row0, (uint32_t)kRows) : 0u;
  const bool own = lane < count;
  float inv = 0.f;
  bool bad = false;
  if (own && !rs.slot_ok && head == 0) raise_error(a.err, ERR_PAGE);
  if (head < a.qh + a.kvh && own) {
    const float sum = qk_square_sum(staged + lane * kQkPitch);
    inv = inverse_rms(sum, 128.0f, a.eps);
    // (A nonfinite element makes the sum nonfinite.)
    bad = !is_finite_f32(sum) | !is_finite_f32(inv);
  }
#pragma unroll 4
  for (uint32_t i = 0; i < kRows / 8; ++i) {
    const uint32_t r = 8 * i + (lane >> 3);
    const float inv_r = __shfl(inv, (int)r);
    const QkvRowSlot rs_r{(uint32_t)__shfl((int)rs.pos, (int)r), (uint32_t)__shfl((int)rs.slot, (int)r),
                          __shfl((int)rs.slot_ok, (int)r) != 0};
    if (r < count) bad |= qknorm_rope_kv_piece(staged + r * kQkPitch, lane & 7u, inv_r, row0 + r, head, a, rs_r);
  }
  if (bad) raise_error(a.err, ERR_NONFINITE);
}

}  // namespace fh
