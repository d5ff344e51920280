// Building blocks of the attention kernels over F16 and BF16 rows (decode and prefill
// chunk): MFMA operands of either type, values split into 16-bit parts, row loads, and the
// shapes the kernels take. Include-only; every symbol has internal linkage.
#pragma once
#include "pkv_mfma_common.hpp"

namespace pkv {

// Scratch of the general kernel's plan: a no-alloc call is accepted when it fits.
size_t generic_plan_bytes(const AttnArgs &a);

namespace {

typedef __bf16 b8 __attribute__((ext_vector_type(8)));

// F16: a weight is at most 2^4 (the running max is raised once a score passes it by 4 in log2
// units) and is held times 2^11, so that its hi + lo is off by 2^-36 at most. With a headroom
// of 2^8 and 2^7, 2^-32: where a first key outweighs the others by e^14 and its V is almost
// nothing, so that the output is made of weights near 2^-20, the error was 2.6e-6 (512 tokens
// over 1536 keys; f32 products 4.5e-7), now 4.5e-7. A headroom of 2 costs 1 to 2% of a
// chunk's time, of 4 under 0.7%.
constexpr float kF16Lazy = 4.0f, kPUp = 2048.0f;
constexpr float kBf16Lazy = 8.0f;

__device__ __forceinline__ float half_value(uint16_t x, bool bf) {
  return bf ? u2f((uint32_t)x << 16) : h2f(x);
}

__device__ __forceinline__ uint32_t bf2(float a, float b) {  // {bf16(a), bf16(b)}, to nearest even
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, b2{(__bf16)a, (__bf16)b});
}
__device__ __forceinline__ float bf_lo(uint32_t w) { return u2f(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return u2f(w & 0xFFFF0000u); }

// The operand words of a pair of values x0, x1 as 16-bit parts: w = the first (lo_col: the
// second), w2 = the third (lo_col: 0). BF16: 8 bits each. F16: 11 bits each, no third (a
// third one of 11 bits, or three of 8, did not change F16's error).
template <bool kBf>
__device__ __forceinline__ void split_pair(float x0, float x1, bool lo_col, uint32_t &w,
                                           uint32_t &w2) {
  const uint32_t mask = lo_col ? 0xFFFFFFFFu : 0u;
  w2 = 0u;
  if constexpr (kBf) {
    const uint32_t h = bf2(x0, x1);
    const float r0 = x0 - bf_lo(h), r1 = x1 - bf_hi(h);
    const uint32_t mid = bf2(r0, r1);
    w = lo_col ? mid : h;
    w2 = bf2(r0 - bf_lo(mid), r1 - bf_hi(mid)) & ~mask;
  } else {
    const h2 h = {(_Float16)x0, (_Float16)x1};
    w = fp16_sub2(x0, x1, as_u(h) & mask);
  }
}
template <bool kBf>
__device__ __forceinline__ f4 half_mfma(u4 a, u4 b, f4 c) {
  if constexpr (kBf)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a),
                                                   __builtin_bit_cast(b8, b), c, 0, 0, 0);
  else
    return mfma32(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c);
}
// The operand negated. The MFMA's sums lose low bits towards minus infinity, a bias of 1/20 of
// the rounding error that a projection of the outputs adds up: every second column is summed
// negated, so that neighbouring columns' biases cancel.
__device__ __forceinline__ u4 half_neg(u4 a) {
  return u4{a.x ^ 0x80008000u, a.y ^ 0x80008000u, a.z ^ 0x80008000u, a.w ^ 0x80008000u};
}
template <typename T>
__device__ __forceinline__ T row_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  if constexpr (sizeof(T) == 16)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}

// kH heads (q rows of 256 floats) over keys [j0, j1) in f32 products, element for element what the
// general kernel (pkv_attn.hip) computes: lane owns elements 4 lane .. + 3; m in log2 units. A
// key's rows are read once for all heads (5 tokens over 20000 keys with NaN: 970 us a head at
// a time, 300 so; the general kernel 570).
template <int kH>
__device__ __forceinline__ void half_slow_keys(const uint8_t *kbase, const uint8_t *vbase,
                                               int64_t rs_t, int64_t j0, int64_t j1, const float *q,
                                               float sl2, bool bf, int lane, float (&m)[kH],
                                               float (&l)[kH], float (&acc)[kH][4]) {
  float4 q4[kH];
#pragma unroll
  for (int h = 0; h < kH; ++h) {
    q4[h] = reinterpret_cast<const float4 *>(q + h * 256)[lane];
    m[h] = -INFINITY;
    l[h] = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[h][k] = 0.0f;
  }
  for (int64_t j = j0; j < j1; ++j) {
    const uint2 kw = *reinterpret_cast<const uint2 *>(kbase + j * rs_t + 8 * lane);
    const uint2 vw = *reinterpret_cast<const uint2 *>(vbase + j * rs_t + 8 * lane);
    const float kf[4] = {half_value((uint16_t)kw.x, bf), half_value((uint16_t)(kw.x >> 16), bf),
                         half_value((uint16_t)kw.y, bf), half_value((uint16_t)(kw.y >> 16), bf)};
    const float vf[4] = {half_value((uint16_t)vw.x, bf), half_value((uint16_t)(vw.x >> 16), bf),
                         half_value((uint16_t)vw.y, bf), half_value((uint16_t)(vw.y >> 16), bf)};
#pragma unroll
    for (int h = 0; h < kH; ++h) {
      float dot = q4[h].x * kf[0];
      dot += q4[h].y * kf[1];
      dot += q4[h].z * kf[2];
      dot += q4[h].w * kf[3];
      const float s = fminf(fmaxf(wave_sum(dot) * sl2, -kClampL2), kClampL2);
      const float mn = fmaxf(m[h], s);
      const float c = __builtin_amdgcn_exp2f(m[h] - mn), p = __builtin_amdgcn_exp2f(s - mn);
      l[h] = l[h] * c + p;
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[h][k] = acc[h][k] * c + p * vf[k];
      m[h] = mn;
    }
  }
}

inline bool half_shape(int quant, int num_heads, int num_kv_heads, int head_dim) {
  return (quant == PKV_QUANT_F16 || quant == PKV_QUANT_BF16) && head_dim == 256 &&
         num_heads == 16 && num_kv_heads == 2;
}
// Scores stay unscaled up to the exponent, so masks and the running max need a positive scale.
inline bool half_scale(float scale) { return scale > 1e-20f && scale < 1e20f; }
// 16-byte loads from every row
inline bool half_aligned(const void *k, const void *v, int64_t rs_b, int64_t rs_t, int64_t rs_h) {
  return ((reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) | (uintptr_t)rs_b |
           (uintptr_t)rs_t | (uintptr_t)rs_h) & 15) == 0 && rs_t > 0 && rs_h >= 0 && rs_b >= 0;
}

}  // namespace
}  // namespace pkv
