// The Q4K superblock quantizer of the throughput kernels (append, prepared append): 8 kL
// lanes per superblock. Include-only; files that include it turn contraction off (every
// a*b+c rounds twice like the Rust code).
#pragma once
#include "pkv_q4k_lanes.hpp"
#include "pkv_scalar.hpp"

namespace pkv {
namespace {

// Lanes per Q4K sub-block in the throughput kernel (kL = 1, 2, 4) and the helpers that
// join a sub-block's kL lanes: all moves within a quad of lanes (DPP), exact.
template <int kL, int q>
__device__ __forceinline__ float group_bcast(float v) {  // lane q of the group's value
  if constexpr (kL == 1) {
    return v;
  } else {
    constexpr int ctrl = kL == 2 ? (q | (q << 2) | ((2 + q) << 4) | ((2 + q) << 6)) : q * 0x55;
    return u2f((uint32_t)__builtin_amdgcn_update_dpp(0, (int)f2u(v), ctrl, 0xF, 0xF, false));
  }
}
template <int kL, typename T, typename Op>
__device__ __forceinline__ T group_allreduce(T v, Op op) {  // order-free ops only
  if constexpr (kL >= 2) {
    const int o = __builtin_amdgcn_update_dpp(0, (int)__builtin_bit_cast(uint32_t, v), 0xB1, 0xF,
                                              0xF, false);  // quad_perm [1,0,3,2]
    v = op(v, __builtin_bit_cast(T, o));
  }
  if constexpr (kL >= 4) {
    const int o = __builtin_amdgcn_update_dpp(0, (int)__builtin_bit_cast(uint32_t, v), 0x4E, 0xF,
                                              0xF, false);  // quad_perm [2,3,0,1]
    v = op(v, __builtin_bit_cast(T, o));
  }
  return v;
}
// acc + term[0] + ... over the whole sub-block, in element order with one rounding per add:
// lane q of the group adds its E terms to the running sum, which every lane then takes
// from lane q (the other lanes' adds that step are discarded).
template <int kL, int q = 0>
struct GroupChain {
  template <int E>
  static __device__ __forceinline__ float run(const float (&term)[E], float acc) {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < E; ++i) acc += term[i];
    acc = group_bcast<kL, q>(acc);
    if constexpr (q + 1 < kL)
      return GroupChain<kL, q + 1>::run(term, acc);
    else
      return acc;
  }
};
template <int kL>
__device__ __forceinline__ bool group_any(bool c) {
  if constexpr (kL == 1) {
    return c;
  } else {
    const uint64_t bal = __ballot(c);
    const int base = (int)(threadIdx.x & 63) & ~(kL - 1);
    return ((bal >> base) & ((1u << kL) - 1)) != 0;
  }
}

// Q4K (BlockQ4K::from_float): 8 kL lanes per 256-element superblock. Lane (j, s) of the
// superblock holds elements [32 j + s E, 32 j + (s + 1) E) of sub-block j, E = 32 / kL.
// The sub-block fit is candle's make_qkx1_quants(nmax = 15, ntry = 5): levels are floats
// (small integers, exact), suml2 an integer-valued f32 (exact, any order), and the two
// other sums run in element order with one rounding per add, lane after lane through the
// group. The element-wise work of a pass is split kL ways and the sums are not, so kL = 1
// gives the fewest instructions per superblock (large appends) and kL = 2 or 4 the
// shortest instruction stream per wave (appends with too few superblocks to fill the GPU).
// Cross-lane work is limited to exact moves, max reductions and byte shuffles.
// r: the lane's index in its superblock's 8 kL (j = r / kL, s = r % kL); block(): the block's 144
// bytes, written where `active` (asked for at the end: an address held through the fit cost
// 2.7% of an append of 4096 tokens, 14.46 us against 14.08).
template <int kL, typename Block>
__device__ __forceinline__ void q4k_quantize_group(const float (&x)[32 / kL], int r, Block block,
                                                   bool active) {
#pragma clang fp contract(off)
  constexpr int E = 32 / kL;
  const int j = r / kL, s = r & (kL - 1);
  // Sub-block min and max in f32::total_cmp order (exact integer keys)
  int32_t kmin = total_key(x[0]), kmax = kmin;
#pragma unroll
  for (int i = 1; i < E; ++i) {
    const int32_t k = total_key(x[i]);
    kmin = k < kmin ? k : kmin;
    kmax = k > kmax ? k : kmax;
  }
  kmin = group_allreduce<kL>(kmin, [](int32_t p, int32_t q) { return p < q ? p : q; });
  kmax = group_allreduce<kL>(kmax, [](int32_t p, int32_t q) { return p > q ? p : q; });
  const auto from_key = [](int32_t k) {
    return u2f((uint32_t)(k ^ (int32_t)(((uint32_t)(k >> 31)) >> 1)));
  };
  const float mn = from_key(kmin), mx = from_key(kmax);

  float scale = 0.0f, mins = 0.0f;
  if (!(mx == mn)) {
    float L[E];
#pragma unroll
    for (int i = 0; i < E; ++i) L[i] = 0.0f;
    float min = fmin_rs(mn, 0.0f);
    float iscale = 15.0f / (mx - min);
    scale = 1.0f / iscale;
    // split fits unroll their passes (no level copies between passes); the one-lane fit
    // stays rolled, unrolled it needs 130 VGPRs and loses a wave per SIMD
    constexpr int kPassUnroll = kL > 1 ? 5 : 1;
#pragma unroll kPassUnroll
    for (int it = 0; it < 5; ++it) {
      float term[E];
      float suml2 = 0.0f;
      bool did_change = false;
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const float d = x[i] - min;
        const float li = (float)q4_level_i(iscale * d);
        did_change |= li != L[i];
        L[i] = li;
        term[i] = d * li;
        suml2 = __builtin_fmaf(li, li, suml2);  // exact
      }
      suml2 = group_allreduce<kL>(suml2, [](float p, float q) { return p + q; });  // exact
      const float sumlx = GroupChain<kL>::run(term, 0.0f);
      scale = sumlx / suml2;
#pragma unroll
      for (int i = 0; i < E; ++i) term[i] = x[i] - scale * L[i];
      const float sum = GroupChain<kL>::run(term, -0.0f);
      min = sum / 32.0f;
      if (min > 0.0f) min = 0.0f;
      iscale = 1.0f / scale;
      if (!group_any<kL>(did_change)) break;
    }
    mins = -min;
  }

  float max_scale = scale, max_min = mins;
#pragma unroll
  for (int o = kL; o < 8 * kL; o <<= 1) {
    max_scale = fmax_rs(max_scale, __shfl_xor(max_scale, o, 8 * kL));
    max_min = fmax_rs(max_min, __shfl_xor(max_min, o, 8 * kL));
  }
  max_scale = fmax_rs(max_scale, 0.0f);
  max_min = fmax_rs(max_min, 0.0f);
  const float inv_scale = max_scale > 0.0f ? 63.0f / max_scale : 0.0f;
  const float inv_min = max_min > 0.0f ? 63.0f / max_min : 0.0f;
  int32_t ls32 = nearest_int(inv_scale * scale);
  int32_t lm32 = nearest_int(inv_min * mins);
  const uint32_t ls = (uint8_t)(ls32 < 63 ? ls32 : 63);
  const uint32_t lm = (uint8_t)(lm32 < 63 ? lm32 : 63);

  const uint16_t dh = f32_to_f16(max_scale / 63.0f);
  const uint16_t mh = f32_to_f16(max_min / 63.0f);

  // get_scale_min_k4(j) of the packed codes returns (ls, lm) for this sub-block.
  // Levels clamp(nearest_int((x + dm) / dd), 0, 15) with a correctly rounded division.
  // Fast path: q = (x + dm) * rcp(dd) is within about 2 ulp of the rounded quotient
  // (v_rcp_f32 within 1 ulp), so rint(q) is its nearest integer unless q lies within
  // 2^-12 of a half-integer (a possible tie); those elements, and every element when
  // rcp(dd) is not finite, take the IEEE division.
  constexpr int NW = (E + 7) / 8;  // nibble words: element i at bits 4 (i % 8) of word i / 8
  uint32_t Lw[NW];
#pragma unroll
  for (int w = 0; w < NW; ++w) Lw[w] = 0u;
  const float dd = f16_to_f32(dh) * (float)ls;
  if (dd != 0.0f) {
    const float dm = f16_to_f32(mh) * (float)lm;
    const float rdd = __builtin_amdgcn_rcpf(dd);
    const bool exact_all = !(__builtin_fabsf(rdd) < 3.0e38f);
    uint32_t slow = 0u;
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const float q = (x[i] + dm) * rdd;
      const float r = __builtin_rintf(q);
      const bool near_tie = __builtin_fabsf(q - r) > 0.5f - 0x1p-12f;
      slow |= (near_tie || exact_all) ? (1u << i) : 0u;
      float l = (r > 0.0f) ? r : 0.0f;  // negatives, -0 and NaN -> 0
      l = (l < 15.0f) ? l : 15.0f;
      Lw[i >> 3] |= (uint32_t)l << (4 * (i & 7));
    }
    if (slow != 0u) {
#pragma unroll
      for (int i = 0; i < E; ++i) {
        if (slow & (1u << i)) {
          const int32_t l = q4_level_i((x[i] + dm) / dd);
          Lw[i >> 3] = (Lw[i >> 3] & ~(15u << (4 * (i & 7)))) | ((uint32_t)l << (4 * (i & 7)));
        }
      }
    }
  }

  // Header: d, dmin, and the 12 packed scale bytes, gathered from the 8 sub-blocks.
  uint32_t code = ls | (lm << 8);
  uint32_t codes[8];
#pragma unroll
  for (int jj = 0; jj < 8; ++jj) codes[jj] = __shfl(code, jj * kL, 8 * kL);
  uint8_t sc[12];
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) {
    const uint32_t ls_lo = codes[jj] & 0xFF, lm_lo = codes[jj] >> 8;
    const uint32_t ls_hi = codes[jj + 4] & 0xFF, lm_hi = codes[jj + 4] >> 8;
    sc[jj] = (uint8_t)(ls_lo | ((ls_hi >> 4) << 6));
    sc[jj + 4] = (uint8_t)(lm_lo | ((lm_hi >> 4) << 6));
    sc[jj + 8] = (uint8_t)((ls_hi & 0xF) | ((lm_hi & 0xF) << 4));
  }

  // Nibbles: qs[32c + l] = L_{2c}[l] | L_{2c+1}[l] << 4. Lanes (2c, s) and (2c+1, s) own
  // l in [sE, sE + E): the even lane writes the first E/2 bytes, the odd lane the rest,
  // each taking the other half of its partner's nibbles (partner: lane ^ kL).
  constexpr int H = E / 2;             // nibbles (= bytes written) per lane
  constexpr int HW = (H + 7) / 8;      // words per half
  const bool odd = (j & 1) != 0;
  uint32_t lo[HW], hi[HW];
#pragma unroll
  for (int w = 0; w < HW; ++w) {
    uint32_t first, second;  // this lane's nibbles [0, H) and [H, E)
    if constexpr (H >= 8) {
      first = Lw[w];
      second = Lw[HW + w];
    } else {
      first = Lw[0] & ((1u << (4 * H)) - 1u);
      second = Lw[0] >> (4 * H);
    }
    const uint32_t recv = __shfl_xor(odd ? first : second, kL, 8 * kL);
    lo[w] = odd ? recv : first;
    hi[w] = odd ? second : recv;
  }
  constexpr int NB = H / 4;  // output words
  uint32_t outw[NB];
#pragma unroll
  for (int w = 0; w < NB; ++w) {
    const uint32_t l4 = lo[w / 2] >> (16 * (w & 1)), h4 = hi[w / 2] >> (16 * (w & 1));
    uint32_t v = 0;
#pragma unroll
    for (int bb = 0; bb < 4; ++bb) {
      const uint32_t ln = (l4 >> (4 * bb)) & 0xF, hn = (h4 >> (4 * bb)) & 0xF;
      v |= (ln | (hn << 4)) << (8 * bb);
    }
    outw[w] = v;
  }
  if (!active) return;
  uint8_t *const blk = block();
  uint8_t *qdst = blk + 16 + 32 * (j >> 1) + s * E + (odd ? H : 0);
  if constexpr (NB == 4) {
    *reinterpret_cast<uint4 *>(qdst) = uint4{outw[0], outw[1], outw[2], outw[3]};
  } else if constexpr (NB == 2) {
    *reinterpret_cast<uint2 *>(qdst) = uint2{outw[0], outw[1]};
  } else {
    *reinterpret_cast<uint32_t *>(qdst) = outw[0];
  }
  if (r == 0) {
    uint4 hd;
    hd.x = (uint32_t)dh | ((uint32_t)mh << 16);
    hd.y = (uint32_t)sc[0] | ((uint32_t)sc[1] << 8) | ((uint32_t)sc[2] << 16) | ((uint32_t)sc[3] << 24);
    hd.z = (uint32_t)sc[4] | ((uint32_t)sc[5] << 8) | ((uint32_t)sc[6] << 16) | ((uint32_t)sc[7] << 24);
    hd.w = (uint32_t)sc[8] | ((uint32_t)sc[9] << 8) | ((uint32_t)sc[10] << 16) | ((uint32_t)sc[11] << 24);
    *reinterpret_cast<uint4 *>(blk) = hd;
  }
}

}  // namespace
}  // namespace pkv
