// MFMA prefill-chunk attention over F16 and BF16 caches of the Qwen3-Next full-attention
// shape (16 query heads, 2 KV heads, head_dim 256), gfx950.
//
// Role: FullAttention::forward for l > 1 over the reference's float cache
// (paramecia-model/src/qwen3_next.rs:2492-2605): the chunk's l queries attend causally over
// every key, scores scaled, clamped to +-100, soft-maxed and applied to V.
//
// Work split, plan and merge are those of the Q4K and Q8_0 chunks (pkv_prefill_common.hpp):
// a workgroup of 8 waves owns one KV head, 16 query positions (two per wave, 8 heads each)
// and one split of the keys. Per 32-key block, waves 4-7 move the K rows into LDS as QK A
// fragments, waves 0-3 the V rows as PV B fragments (pairs of keys joined by v_perm), each
// a block ahead through registers; all waves then run QK and PV from LDS, one barrier per
// block. Bound: the MFMAs (F16 two per operand, BF16 three) and the softmax between them.
// Before, such chunks ran the general kernel (one wave reduction per key and head): us,
// F16 (l queries over S keys): 2 x 64 54.7 to 11.3; 5 x 1000 60.9 to 15.6; 5 x 20016 567 to
// 24.5; 16 x 4000 311 to 26.6; 100 x 600 232 to 25.5; 512 x 1024 1750 to 42. BF16: 48 to
// 12.1, 54 to 15.1, 538 to 27, 292 to 29, 215 to 28, 1632 to 47.
//
// Precision and non-finite values as in the decode (pkv_half_decode.hip): q and p enter as
// sums of 16-bit parts; a wave that meets infinities or NaN redoes its rows in f32. Mean
// error against 64 bits over 7 x 64 to 100 x 3000, scores of standard deviation 0.01 to 12:
// 0.44 to 1.08 times the general kernel's (7 x 5007, 1: F16 2.0e-7 of 3.6e-7).
#include "pkv_half_common.hpp"
#include "pkv_prefill_common.hpp"

namespace pkv {
namespace {

struct HalfBlock {
  // QK A: [tile][step], lane (r, g) at 16 g + (r ^ ((4 step + g) % 16)): the pieces of a row,
  // written by 32 lanes at once, then lie on different banks
  u4 ka[2][8][64];
  u4 vb[16][64];    // PV B: tile 4 w + j, column n: e = 64 w + 4 n + j
};
struct HalfPfSmem {
  HalfBlock blk[2];  // block i in blk[i & 1] while block i + 1 is written
};

// A wave's rows (positions pw, pw + 1) over keys [k0, k1) in f32 products. Writes the rows'
// outputs or partials.
__device__ __forceinline__ void slow_wave(const PrefillArgs &a, const uint8_t *kbase,
                                          const uint8_t *vbase, int64_t k0, int64_t k1, int pw,
                                          int b, int kvg, int64_t r0, bool bf, int lane) {
  for (int pos = pw; pos < pw + 2 && pos < a.l; ++pos) {
    const int64_t qr = ((int64_t)b * a.l + pos) * 16 + 8 * kvg;
    const int64_t lim = a.causal ? pos + a.q_offset + 1 : a.seq_k;
    float m[8], l[8], acc[8][4];
    half_slow_keys<8>(kbase, vbase, a.rs_t, k0, lim < k1 ? lim : k1, a.q + qr * 256, a.sl2, bf, lane,
                      m, l, acc);
#pragma unroll
    for (int h = 0; h < 8; ++h) {
      if (a.nsplit == 1) {
        const float inv = l[h] > 0.0f ? 1.0f / l[h] : 0.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k) a.out[(qr + h) * 256 + 4 * lane + k] = acc[h][k] * inv;
      } else {
        const int64_t r = r0 + (int64_t)pos * 8 + h;
#pragma unroll
        for (int k = 0; k < 4; ++k) a.part[r * 256 + tile_index(4 * lane + k)] = acc[h][k];
        if (lane == 0) a.ml[r] = float2{m[h], l[h]};
      }
    }
  }
}

template <bool kBf>
__global__ __launch_bounds__(kPfThreads) void half_prefill_kernel(PrefillArgs a) {
  __shared__ HalfPfSmem sm;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const PfWork wk = prefill_work(a);
  const int tile = wk.tile, kvg = wk.kvg, split = wk.split, b = wk.b;
  const int p0 = tile * kPosPerWG;
  const int pw = p0 + 2 * wave;  // this wave's first position (row n -> pw + n / 8)
  const bool active = pw < a.l;

  int64_t kend = a.seq_k;
  if (a.causal) {
    const int64_t plast = (p0 + kPosPerWG - 1 < a.l ? p0 + kPosPerWG - 1 : a.l - 1);
    const int64_t lim = plast + a.q_offset + 1;
    if (lim < kend) kend = lim;
  }
  const int nblk_all = (int)((kend + kBlk - 1) / kBlk);
  const int bps = (nblk_all + a.nsplit - 1) / a.nsplit;
  const int kb0 = split * bps;
  const int kb1 = kb0 + bps < nblk_all ? kb0 + bps : nblk_all;
  const int nb = kb1 > kb0 ? kb1 - kb0 : 0;

  const uint8_t *kbase = a.k + b * a.rs_b + kvg * a.rs_h;
  const uint8_t *vbase = a.v + b * a.rs_b + kvg * a.rs_h;
  const uint32_t rs_t = (uint32_t)a.rs_t;
  const int last = (int)a.seq_k - 1;  // loads past it read the last row again (masked)
  const uint32_t span = a.seq_k > 0 ? (uint32_t)last * rs_t + 512u : 0u;
  const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t *>(wave >= 4 ? kbase : vbase), 0, span, 0x00020000);
  // Waves 4-7: 16-byte piece c of key 8 (wave - 4) + 2 i + lane / 32 (c = lane % 32); waves
  // 0-3: 8 bytes (columns 64 wave + 4 n .. + 3) of keys 8 g + 2 i and + 1, as one pair.
  u4 st[4];
  auto load = [&](int blk) {
    if (wave >= 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = blk * kBlk + 8 * (wave - 4) + 2 * i + (lane >> 5);
        st[i] = row_load<u4>(rows, (uint32_t)(key < last ? key : last) * rs_t + 16u * (lane & 31));
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k0 = blk * kBlk + 8 * g + 2 * i;
        const uint2 x = row_load<uint2>(rows, (uint32_t)(k0 < last ? k0 : last) * rs_t + 128u * wave + 8u * n);
        const uint2 y = row_load<uint2>(rows, (uint32_t)(k0 + 1 < last ? k0 + 1 : last) * rs_t + 128u * wave + 8u * n);
        st[i] = u4{x.x, x.y, y.x, y.y};
      }
    }
  };
  auto store = [&](HalfBlock &D) {
    if (wave >= 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {  // key kk is row r of tile t: kk = 8 (r / 4) + 4 t + r % 4
        const int kk = 8 * (wave - 4) + 2 * i + (lane >> 5), c = lane & 31;
        const int t = (kk >> 2) & 1, r = 4 * (kk >> 3) + (kk & 3);
        D.ka[t][c >> 2][16 * (c & 3) + (r ^ (c & 15))] = st[i];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          w[i] = j < 2 ? __builtin_amdgcn_perm(st[i].z, st[i].x, sel)
                       : __builtin_amdgcn_perm(st[i].w, st[i].y, sel);
        D.vb[4 * wave + j][lane] = u4{w[0], w[1], w[2], w[3]};
      }
    }
  };
  if (nb > 0) load(kb0);

  // ---- q operands of this wave's 16 rows: lane (n, g) holds elements 32 s + 8 g .. + 7
  u4 qh[8], ql[8], q3[kBf ? 8 : 1];
  float cs = a.sl2;
  {
    const int pos = pw + (n >> 3);
    // rows past the chunk read position 0 and are never stored
    const float *qrow = a.q + (((int64_t)b * a.l + (pos < a.l ? pos : 0)) * 16 + 8 * kvg + (n & 7)) * 256 + 8 * g;
    float4 v[8][2];
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int x = 0; x < 2; ++x) v[s][x] = *reinterpret_cast<const float4 *>(qrow + 32 * s + 4 * x);
    float f = 1.0f;
    if constexpr (!kBf) {  // the row to [2^14, 2^15)
      float mx = 0.0f;
#pragma unroll
      for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int x = 0; x < 2; ++x)
          mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[s][x].x), fabsf(v[s][x].y)),
                               fmaxf(fabsf(v[s][x].z), fabsf(v[s][x].w))));
      mx = xmax32(xmax16(mx));
      int e = (int)(f2u(mx) >> 23) - 127;
      e = e < -100 ? -100 : e > 100 ? 100 : e;
      f = __builtin_ldexpf(1.0f, 14 - e);
      cs = a.sl2 * __builtin_ldexpf(1.0f, e - 14);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      uint32_t w1[4], w2[4], w3[4], none;
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const float fs = (s & 1) ? -f : f;  // odd s are summed negated, as the odd columns
        const float y[4] = {v[s][x].x * fs, v[s][x].y * fs, v[s][x].z * fs, v[s][x].w * fs};
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          split_pair<kBf>(y[2 * k], y[2 * k + 1], false, w1[2 * x + k], w3[2 * x + k]);
          split_pair<kBf>(y[2 * k], y[2 * k + 1], true, w2[2 * x + k], none);
        }
      }
      qh[s] = u4{w1[0], w1[1], w1[2], w1[3]};
      ql[s] = u4{w2[0], w2[1], w2[2], w2[3]};
      if constexpr (kBf) q3[s] = u4{w3[0], w3[1], w3[2], w3[3]};
    }
  }

  const f4 zero = {0.f, 0.f, 0.f, 0.f};
  f4 acc[16];
#pragma unroll
  for (int T = 0; T < 16; ++T) acc[T] = zero;
  constexpr float kUp = kBf ? 1.0f : kPUp;  // (not in the exponents: it would round them)
  const float clamp = kClampL2 / cs, lazy = (kBf ? kBf16Lazy : kF16Lazy) / cs;
  float m_run = -INFINITY, nm = INFINITY, lsum = 0.0f;
  bool bad = false;
  const int64_t klim = a.causal ? (int64_t)pw + (n >> 3) + a.q_offset : (int64_t)1 << 62;
  if (nb > 0) {
    store(sm.blk[0]);
    if (nb > 1) load(kb0 + 1);
  }
  for (int i = 0; i < nb; ++i) {
    lds_barrier();  // block i is in LDS; block i - 1 is no longer read
    if (i + 1 < nb) {
      store(sm.blk[(i + 1) & 1]);
      if (i + 2 < nb) load(kb0 + i + 2);
    }
    if (!active) continue;
    const HalfBlock &D = sm.blk[i & 1];
    // ---- QK: keys kk of the block at or past nlim are masked (past the cache, or past this
    // row's causal limit)
    int64_t lim = a.seq_k < klim + 1 ? a.seq_k : klim + 1;
    lim -= (int64_t)(kb0 + i) * kBlk;
    const int nlim = lim < 0 ? 0 : (lim > kBlk ? kBlk : (int)lim);
    // (short chains, summed as a tree: one chain of 8 accumulations per part had 1.5 times
    // the general kernel's error)
    float sc8[8], ca[8], cb[8], big = 0.0f;  // sc8 = ca + cb, rounded
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f4 c[4] = {zero, zero, zero, zero}, r[2] = {zero, zero};
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const u4 A = D.ka[t][s][16 * g + (n ^ ((4 * s + g) & 15))];
        c[s & 3] = half_mfma<kBf>(A, qh[s], c[s & 3]);
        r[s & 1] = half_mfma<kBf>(A, ql[s], r[s & 1]);
        if constexpr (kBf) r[s & 1] = half_mfma<kBf>(A, q3[s], r[s & 1]);
      }
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const int k = 4 * t + ii, kk = 8 * g + k;
        ca[k] = c[0][ii] - c[1][ii];
        cb[k] = (c[2][ii] - c[3][ii]) + (r[0][ii] - r[1][ii]);
        const float sc = ca[k] + cb[k];
        bad |= kk < nlim && !(fabsf(sc) < INFINITY);
        sc8[k] = kk < nlim ? sc : -INFINITY;
        big = fmaxf(big, kk < nlim ? fabsf(sc) : 0.0f);
      }
    }
    if (__any(big > clamp)) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (!(fabsf(sc8[k]) > clamp) || sc8[k] == -INFINITY) continue;
        sc8[k] = ca[k] = __builtin_amdgcn_fmed3f(sc8[k], -clamp, clamp);
        cb[k] = 0.0f;
      }
    }
    // ---- online softmax per row (lanes n, n + 16, n + 32, n + 48 hold row n's 32 keys)
    float bm = sc8[0];
#pragma unroll
    for (int k = 1; k < 8; ++k) bm = fmaxf(bm, sc8[k]);
    bm = xmax32(xmax16(bm));
    if (__any(bm > m_run + lazy)) {
      const float m_new = fmaxf(m_run, bm);
      const float nm_new = m_new == -INFINITY ? INFINITY : -(m_new * cs);
      const float alpha = (m_run == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(nm_new - nm);
      lsum *= alpha;
      m_run = m_new;
      nm = nm_new;
      float ai[4];
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) ai[ii] = __shfl(alpha, 4 * g + ii);  // rows 4g+ii
#pragma unroll
      for (int T = 0; T < 16; ++T)
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) acc[T][ii] *= ai[ii];
    }
    float p[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      // (the score's two summands one after the other: where p is large the sums are small, and
      // the rounding of sc8, up to 2^-21 of it, does not enter)
      const float e = fmaf(cb[k], cs, fmaf(ca[k], cs, nm));
      p[k] = sc8[k] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(e) * kUp;
      lsum += p[k];
    }
    // ---- PV: A rows = query rows, keys 8 g .. 8 g + 7
    uint32_t w1[4], w2[4], w3[4], none;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      split_pair<kBf>(p[2 * k], p[2 * k + 1], false, w1[k], w3[k]);
      split_pair<kBf>(p[2 * k], p[2 * k + 1], true, w2[k], none);
    }
    const u4 A = {w1[0], w1[1], w1[2], w1[3]}, Al = {w2[0], w2[1], w2[2], w2[3]};
    const u4 A3 = {w3[0], w3[1], w3[2], w3[3]};
    const u4 An = half_neg(A), Aln = half_neg(Al), A3n = half_neg(A3);  // odd columns
#pragma unroll
    for (int T = 0; T < 16; ++T) {
      const u4 B = D.vb[T][lane];
      acc[T] = half_mfma<kBf>((T & 1) ? An : A, B, acc[T]);
      acc[T] = half_mfma<kBf>((T & 1) ? Aln : Al, B, acc[T]);
      if constexpr (kBf) acc[T] = half_mfma<kBf>((T & 1) ? A3n : A3, B, acc[T]);
    }
  }
  if (!active) return;

  // ---- epilogue: row sums, then the output or the split's partial
  lsum += __shfl_xor(lsum, 16);
  lsum += __shfl_xor(lsum, 32);
  const int64_t r0 = ((int64_t)(b * a.nsplit + split) * 2 + kvg) * a.l * 8;
#pragma unroll
  for (int T = 0; T < 16; ++T)
#pragma unroll
    for (int ii = 0; ii < 4; ++ii)
      bad |= pw + ((4 * g + ii) >> 3) < a.l && !(fabsf(acc[T][ii]) < INFINITY);
  if (__any(bad)) {
    const int64_t k1 = (int64_t)kb1 * kBlk < a.seq_k ? (int64_t)kb1 * kBlk : a.seq_k;
    slow_wave(a, kbase, vbase, (int64_t)kb0 * kBlk, k1, pw, b, kvg, r0, kBf, lane);
    return;
  }
  const float mx = -nm;  // log2 units
#pragma unroll
  for (int ii = 0; ii < 4; ++ii) {  // m and l of row 4g+ii live in lane 4g+ii (any g)
    const float lrow = __shfl(lsum, 4 * g + ii), mrow = __shfl(mx, 4 * g + ii);
    const int row = 4 * g + ii, pos = pw + (row >> 3);
    if (pos >= a.l) continue;
    if (a.nsplit == 1) {
      float *orow = a.out + (((int64_t)b * a.l + pos) * 16 + 8 * kvg + (row & 7)) * 256;
      const float inv = lrow > 0.0f ? 1.0f / lrow : 0.0f;
#pragma unroll
      for (int w = 0; w < 4; ++w)
        *reinterpret_cast<float4 *>(orow + 64 * w + 4 * n) =
            float4{acc[4 * w][ii] * inv, acc[4 * w + 1][ii] * -inv, acc[4 * w + 2][ii] * inv,
                   acc[4 * w + 3][ii] * -inv};
    } else {
      const int64_t r = r0 + (int64_t)pos * 8 + (row & 7);
#pragma unroll
      for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          a.part[r * 256 + tile_index(64 * w + 4 * n + j)] =
              acc[4 * w + j][ii] * ((j & 1) ? -1.0f / kUp : 1.0f / kUp);
      if (n == 0) a.ml[r] = float2{mrow, lrow * (1.0f / kUp)};
    }
  }
}

}  // namespace

int launch_prefill_half(const AttnArgs &a, Workspace &ws, hipStream_t s) {
  if (!half_shape(a.quant, a.num_heads, a.num_kv_heads, a.head_dim) || a.l < 2)
    return PKV_ERR_UNSUPPORTED;
  if (!half_scale(a.scale) || !half_aligned(a.k, a.v, a.rs.b, a.rs.t, a.rs.h) || !decode_rows_fit(a.seq_k, a.rs.t) ||
      ((reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.out)) & 15) != 0)
    return PKV_ERR_UNSUPPORTED;
  const bool bf = a.quant == PKV_QUANT_BF16;
  return prefill_run(a, a.scale * kLog2e, ws, s, generic_plan_bytes(a), [&](const PrefillArgs &d, dim3 grid) {
    if (bf)
      hipLaunchKernelGGL(half_prefill_kernel<true>, grid, dim3(kPfThreads), 0, s, d);
    else
      hipLaunchKernelGGL(half_prefill_kernel<false>, grid, dim3(kPfThreads), 0, s, d);
  });
}

}  // namespace pkv
