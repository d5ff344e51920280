// MFMA decode attention over F16 and BF16 caches of the Qwen3-Next full-attention shape
// (16 query heads, 2 KV heads, head_dim 256), gfx950.
//
// Role: the CPU SDPA of the reference's float cache (paramecia-model/src/qwen3_next.rs:
// 2492-2605) for a decode step: every query head reads the keys of KV head h / 8, scores
// scaled, clamped to +-100, soft-maxed and applied to V.
//
// Bound: HBM, 2048 bytes per cached key. No LDS in the loop: a row's halves are MFMA
// operands as they are. A workgroup of 4 waves owns a range of 32-key blocks of one
// segment (a cache's batch row, or a sequence); wave w takes KV head w % 2 of every second
// block, and reads
//   K as A operands: lane (r, g) takes key kk(r, t), elements 32 s + 8 g .. + 7 (16 bytes);
//   V as whole 256-byte half rows: lane (n, g) takes elements 128 u + 8 n .. + 7 of keys
//   8 g .. 8 g + 7, and pairs of keys become B operands with one v_perm per pair and
//   column: tile 8 u + j holds columns e = 128 u + 8 n + j.
// Keys are permuted inside a block so that the QK result layout is the PV A layout. The
// new token of a fused step is converted by the first workgroups and joins in the combine
// (pkv_decode_split.hpp) from its rounded rows.
// 12290 keys, one layer (25.2 MB): append, general kernel and combine took 160 us; this
// kernel and its combine take 15.9 us (131073 keys, 268 MB: 56.7 us, 4.7 TB/s). Below 4096
// keys the 14.4 us are the chain of one block's latencies. Tried: 512 workgroups instead
// of 256 (32.8 against 22.1 us at 32768 keys: the combine reads twice the partials), V
// read ahead by a block (16.8 us at 12290).
//
// Precision: q and the weights p enter as sums of 16-bit parts, accumulated in f32: F16 hi
// and lo (q scaled by a power of two per row, p by 2^7, so that neither part leaves fp16's
// range: 22 bits), BF16 three parts (24 bits).
//
// Infinities and NaN (a float cache stores what it is given; F16 overflows to infinity):
// a split operand times infinity can give inf - inf, so a wave whose scores or sums come
// out non-finite redoes its blocks in plain f32 products (slow_rows), element for element
// what the general kernel (pkv_attn.hip) computes.
#include "pkv_decode_split.hpp"
#include "pkv_mfma_common.hpp"

namespace pkv {

// The no-alloc entry accepts a call when the general kernel's plan fits its scratch.
int generic_plan_fits(const AttnArgs &a, Workspace &ws);

namespace {

typedef __bf16 b8 __attribute__((ext_vector_type(8)));

constexpr int kHdWaves = 4, kHdThreads = 64 * kHdWaves;
constexpr int kHdTargetWGs = 256;  // partial slots of a full launch
constexpr float kHdLazy = 8.0f;    // log2 headroom of the running max before a rescale
constexpr float kPBias = 7.0f;     // F16: p is held times 2^7 (at most 2^15 with the headroom)

struct HalfSeg {
  uint8_t *k, *v;  // rows of token 0, KV head 0
  int64_t seq_k;   // keys attended here (a fused step's new key joins in the combine)
  int64_t t_new;   // row the fused step writes
  int nblk, wg0, nwg;
};
template <int kSegs>
struct HalfArgs {
  int64_t rs_t, rs_h;
  int nseg, fused;
  float sl2;                   // scale * log2(e)
  const float *q;              // [nseg][16][256]
  const float *k_new, *v_new;  // [nseg][2][256]
  float *part;                 // [slot][16][256] in tile order
  float2 *ml;                  // [slot][16]
  float *dq;                   // [nseg][4][256]
  HalfSeg seg[kSegs];
};

struct HalfSmem {
  float o[kHdWaves][8][256];
  float m[kHdWaves][8], l[kHdWaves][8];
};

__device__ __forceinline__ float half_value(uint16_t x, bool bf) {
  return bf ? u2f((uint32_t)x << 16) : h2f(x);
}

// One wave's blocks in f32 products (see the header): lane owns elements 4 lane .. + 3.
__device__ __forceinline__ void slow_rows(const uint8_t *kbase, const uint8_t *vbase,
                                          int64_t rs_t, int64_t seq_k, int first, int step,
                                          int last, const float *q, float sl2, bool bf, int lane,
                                          float (*o)[256], float *mo, float *lo) {
  for (int h = 0; h < 8; ++h) {
    const float4 q4 = reinterpret_cast<const float4 *>(q + h * 256)[lane];
    float m = -INFINITY, l = 0.0f, acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int b = first; b < last; b += step) {
      const int64_t k1 = (int64_t)(b + 1) * kBlk < seq_k ? (int64_t)(b + 1) * kBlk : seq_k;
      for (int64_t j = (int64_t)b * kBlk; j < k1; ++j) {
        const uint2 kw = *reinterpret_cast<const uint2 *>(kbase + j * rs_t + 8 * lane);
        const uint2 vw = *reinterpret_cast<const uint2 *>(vbase + j * rs_t + 8 * lane);
        float part = q4.x * half_value((uint16_t)kw.x, bf);
        part += q4.y * half_value((uint16_t)(kw.x >> 16), bf);
        part += q4.z * half_value((uint16_t)kw.y, bf);
        part += q4.w * half_value((uint16_t)(kw.y >> 16), bf);
        const float s = fminf(fmaxf(wave_sum(part) * sl2, -kClampL2), kClampL2);
        const float mn = fmaxf(m, s);
        const float c = __builtin_amdgcn_exp2f(m - mn), p = __builtin_amdgcn_exp2f(s - mn);
        l = l * c + p;
        acc[0] = acc[0] * c + p * half_value((uint16_t)vw.x, bf);
        acc[1] = acc[1] * c + p * half_value((uint16_t)(vw.x >> 16), bf);
        acc[2] = acc[2] * c + p * half_value((uint16_t)vw.y, bf);
        acc[3] = acc[3] * c + p * half_value((uint16_t)(vw.y >> 16), bf);
        m = mn;
      }
    }
    *reinterpret_cast<float4 *>(&o[h][4 * lane]) = float4{acc[0], acc[1], acc[2], acc[3]};
    if (lane == 0) {
      mo[h] = m;
      lo[h] = l;
    }
  }
}

__device__ __forceinline__ uint32_t bf2(float a, float b) {  // {bf16(a), bf16(b)}, to nearest even
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, b2{(__bf16)a, (__bf16)b});
}
__device__ __forceinline__ float bf_lo(uint32_t w) { return u2f(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return u2f(w & 0xFFFF0000u); }

// The operand words of a pair of values x0, x1. F16: w = the hi parts (lo_col: the lo
// remainders). BF16: w = the first parts (lo_col: the second), w2 = the third (lo_col: 0).
template <bool kBf>
__device__ __forceinline__ void split_pair(float x0, float x1, bool lo_col, uint32_t &w,
                                           uint32_t &w2) {
  const uint32_t mask = lo_col ? 0xFFFFFFFFu : 0u;
  if constexpr (kBf) {
    const uint32_t h = bf2(x0, x1);
    const float r0 = x0 - bf_lo(h), r1 = x1 - bf_hi(h);
    const uint32_t mid = bf2(r0, r1);
    const uint32_t third = bf2(r0 - bf_lo(mid), r1 - bf_hi(mid));
    w = lo_col ? mid : h;
    w2 = third & ~mask;
  } else {
    w = fp16_sub2(x0, x1, as_u(h2{(_Float16)x0, (_Float16)x1}) & mask);
    w2 = 0u;
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
__device__ __forceinline__ u4 row16(__amdgpu_buffer_rsrc_t r, uint32_t off, int imm) {
  return __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(r, off + imm, 0, 0));
}

template <bool kBf, int kSegs>
__global__ __launch_bounds__(kHdThreads) void half_decode_kernel(HalfArgs<kSegs> a) {
  __shared__ HalfSmem sm;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kv = wave & 1, sub = wave >> 1;
  int s = 0;
  if constexpr (kSegs > 1)
    while (s + 1 < a.nseg && a.seg[s + 1].wg0 <= (int)blockIdx.x) ++s;
  const HalfSeg sg = a.seg[s];
  // blocks [b0, b1) of the segment
  const int w = (int)blockIdx.x - sg.wg0, bq = sg.nblk / sg.nwg, br = sg.nblk % sg.nwg;
  const int b0 = w * bq + (w < br ? w : br), b1 = b0 + bq + (w < br ? 1 : 0);
  const uint32_t rs_t = (uint32_t)a.rs_t;
  const uint8_t *kbase = sg.k + kv * a.rs_h, *vbase = sg.v + kv * a.rs_h;
  const int last = (int)sg.seq_k - 1;  // loads past it read the last row again (masked)
  const uint32_t span = sg.seq_k > 0 ? (uint32_t)last * rs_t + 512u : 0u;
  const __amdgpu_buffer_rsrc_t rk =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(kbase), 0, span, 0x00020000);
  const __amdgpu_buffer_rsrc_t rv =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(vbase), 0, span, 0x00020000);
  u4 kw[2][8], vw[8][2];
  auto load_k = [&](int b) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int key = b * kBlk + 8 * (n >> 2) + 4 * t + (n & 3);
      const uint32_t off = (uint32_t)(key < last ? key : last) * rs_t + 16u * g;
#pragma unroll
      for (int st = 0; st < 8; ++st) kw[t][st] = row16(rk, off, 64 * st);
    }
  };
  auto load_v = [&](int b) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int key = b * kBlk + 8 * g + k;
      const uint32_t off = (uint32_t)(key < last ? key : last) * rs_t + 16u * n;
      vw[k][0] = row16(rv, off, 0);
      vw[k][1] = row16(rv, off, 256);
    }
  };
  const int first = b0 + sub;
  const float *qseg = a.q + ((int64_t)s * 16 + 8 * kv) * 256;
  // q operands: lane (n, g) holds elements 32 st + 8 g .. + 7 of head n % 8
  float4 qv[8][2];
#pragma unroll
  for (int st = 0; st < 8; ++st)
#pragma unroll
    for (int x = 0; x < 2; ++x)
      qv[st][x] = *reinterpret_cast<const float4 *>(qseg + (n & 7) * 256 + 32 * st + 8 * g + 4 * x);
  if (first < b1) {
    load_k(first);
  }

  // Fused step: row 4 i + 2 p + kv (segment i, K (p = 0) or V) is converted and stored
  if (a.fused) {
    for (int row = blockIdx.x; row < 4 * a.nseg; row += gridDim.x) {
      const int i = row >> 2, p = (row >> 1) & 1, h = row & 1;
      const float x = (p ? a.v_new : a.k_new)[((int64_t)i * 2 + h) * 256 + tid];
      const uint16_t y = kBf ? f32_to_bf16(x) : f32_to_f16(x);
      const HalfSeg &r = a.seg[kSegs > 1 ? i : 0];
      reinterpret_cast<uint16_t *>((p ? r.v : r.k) + r.t_new * a.rs_t + h * a.rs_h)[tid] = y;
      a.dq[(int64_t)row * 256 + tid] = half_value(y, kBf);
    }
  }

  u4 qb[8], qb2[8];
  float cs = a.sl2;  // a score is its MFMA result * cs, in log2 units
  float f = 1.0f;
  if constexpr (!kBf) {  // q to [2^14, 2^15)
    float mx = 0.0f;
#pragma unroll
    for (int st = 0; st < 8; ++st)
#pragma unroll
      for (int x = 0; x < 2; ++x)
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(qv[st][x].x), fabsf(qv[st][x].y)),
                             fmaxf(fabsf(qv[st][x].z), fabsf(qv[st][x].w))));
    mx = xmax32(xmax16(mx));
    int e = (int)(f2u(mx) >> 23) - 127;
    e = e < -100 ? -100 : e > 100 ? 100 : e;
    f = __builtin_ldexpf(1.0f, 14 - e);
    cs = a.sl2 * __builtin_ldexpf(1.0f, e - 14);
  }
#pragma unroll
  for (int st = 0; st < 8; ++st) {
    uint32_t w1[4], w2[4];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      split_pair<kBf>(qv[st][x].x * f, qv[st][x].y * f, n >= 8, w1[2 * x], w2[2 * x]);
      split_pair<kBf>(qv[st][x].z * f, qv[st][x].w * f, n >= 8, w1[2 * x + 1], w2[2 * x + 1]);
    }
    qb[st] = u4{w1[0], w1[1], w1[2], w1[3]};
    qb2[st] = u4{w2[0], w2[1], w2[2], w2[3]};
  }

  const f4 zero = {0.f, 0.f, 0.f, 0.f};
  f4 acc[16];
#pragma unroll
  for (int T = 0; T < 16; ++T) acc[T] = zero;
  // Scores and the running max stay in MFMA units; the scale enters the exponents as one
  // fma (rounding a score of tens of log2 units instead cost 2-4 times the error where a
  // few keys dominate). nm: log2 of the weights' common factor.
  constexpr float kBias = kBf ? 0.0f : kPBias;
  const float clamp = kClampL2 / cs, lazy = kHdLazy / cs;
  float m_run = -INFINITY, nm = INFINITY, lsum = 0.0f;
  bool bad = false;
  for (int b = first; b < b1; b += 2) {
    load_v(b);
    // ---- scores of keys 8 g + 4 t + i, head n % 8 (hi columns n < 8, lo columns n >= 8)
    float sc8[8];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f4 c0 = zero, c1 = zero;
#pragma unroll
      for (int st = 0; st < 8; st += 2) {
        c0 = half_mfma<kBf>(kw[t][st], qb[st], c0);
        c1 = half_mfma<kBf>(kw[t][st + 1], qb[st + 1], c1);
        if constexpr (kBf) {
          c0 = half_mfma<kBf>(kw[t][st], qb2[st], c0);
          c1 = half_mfma<kBf>(kw[t][st + 1], qb2[st + 1], c1);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float part = c0[i] + c1[i];
        const float sum = part + ror8(part);
        bad |= !(fabsf(sum) < INFINITY);
        sc8[4 * t + i] = __builtin_amdgcn_fmed3f(sum, -clamp, clamp);
      }
    }
    if (b + 2 < b1) load_k(b + 2);
    const int nvalid = (int)sg.seq_k - b * kBlk;
    if (nvalid < kBlk) {
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (8 * g + k >= nvalid) sc8[k] = -INFINITY;
    }
    // ---- online softmax (lanes n, n + 16, n + 32, n + 48 hold a head's 32 keys)
    float bm = sc8[0];
#pragma unroll
    for (int k = 1; k < 8; ++k) bm = fmaxf(bm, sc8[k]);
    bm = xmax32(xmax16(bm));
    if (m_run == -INFINITY) {
      m_run = bm;
      nm = kBias - bm * cs;
    } else if (__any(bm > m_run + lazy)) {
      m_run = fmaxf(m_run, bm);
      const float nm_new = kBias - m_run * cs;
      const float alpha = __builtin_amdgcn_exp2f(nm_new - nm);
      lsum *= alpha;
      nm = nm_new;
      float ai[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) ai[i] = __shfl(alpha, 4 * (g & 1) + i);
#pragma unroll
      for (int T = 0; T < 16; ++T)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[T][i] *= ai[i];
    }
    float p[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      p[k] = __builtin_amdgcn_exp2f(fmaf(sc8[k], cs, nm));
      lsum += p[k];
    }
    u4 A, A2;
    {
      uint32_t w1[4], w2[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) split_pair<kBf>(p[2 * k], p[2 * k + 1], n >= 8, w1[k], w2[k]);
      A = u4{w1[0], w1[1], w1[2], w1[3]};
      A2 = u4{w2[0], w2[1], w2[2], w2[3]};
    }
    // ---- PV: tile 8 u + j, column n: e = 128 u + 8 n + j
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
        uint32_t bw[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          bw[k] = __builtin_amdgcn_perm(vw[2 * k + 1][u][j >> 1], vw[2 * k][u][j >> 1], sel);
        const u4 B = {bw[0], bw[1], bw[2], bw[3]};
        acc[8 * u + j] = half_mfma<kBf>(A, B, acc[8 * u + j]);
        if constexpr (kBf) acc[8 * u + j] = half_mfma<kBf>(A2, B, acc[8 * u + j]);
      }
  }

  // ---- this wave's rows into LDS: rows h and h + 8 summed (lanes 0-31 keep the columns of
  // u = 0, lanes 32-63 those of u = 1), heads 4 (g & 1) + i
  lsum += __shfl_xor(lsum, 16);
  lsum += __shfl_xor(lsum, 32);
  const int gr = g & 1, u = g >> 1;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float r[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      r[j] = pair_sum32(acc[j][i], acc[8 + j][i]);
      bad |= !(fabsf(r[j]) < INFINITY);
    }
    float *o = &sm.o[wave][4 * gr + i][128 * u + 8 * n];
    reinterpret_cast<float4 *>(o)[0] = float4{r[0], r[1], r[2], r[3]};
    reinterpret_cast<float4 *>(o)[1] = float4{r[4], r[5], r[6], r[7]};
  }
  if (lane < 8) {
    sm.m[wave][n] = -nm;
    sm.l[wave][n] = lsum;
  }
  if (__any(bad))
    slow_rows(kbase, vbase, a.rs_t, sg.seq_k, first, 2, b1, qseg, a.sl2, kBf, lane, sm.o[wave],
              sm.m[wave], sm.l[wave]);
  __syncthreads();
  // ---- the two waves of each KV head merged into the workgroup's partial, in tile order
  const int e = tile_e(tid >> 4, tid & 15);
#pragma unroll
  for (int h = 0; h < 16; ++h) {
    const int w0 = h >> 3, w1 = w0 + 2, r = h & 7;
    const float m0 = sm.m[w0][r], m1 = sm.m[w1][r], M = fmaxf(m0, m1);
    float v = 0.0f, L = 0.0f;
    if (m0 != -INFINITY) {
      const float c = __builtin_amdgcn_exp2f(m0 - M);
      v = sm.o[w0][r][e] * c;
      L = sm.l[w0][r] * c;
    }
    if (m1 != -INFINITY) {
      const float c = __builtin_amdgcn_exp2f(m1 - M);
      v += sm.o[w1][r][e] * c;
      L += sm.l[w1][r] * c;
    }
    const int64_t slot = (int64_t)blockIdx.x * 16 + h;
    __builtin_nontemporal_store(v, a.part + slot * kPartRow + tid);
    if (tid == 0) a.ml[slot] = float2{M, L};
  }
}

// Plan and launch the decode and the combine over n <= kMaxSegs segments. Every segment
// gets workgroups in proportion to its blocks, at most one per two blocks (a block per
// wave pair) and kHdTargetWGs in all (and at least one each).
int launch_half_segments(int quant, const DecodeSegIn *in, int n, const float *q,
                         const float *k_new, const float *v_new, float *out, int64_t rs_t,
                         int64_t rs_h, float scale, Workspace &ws, hipStream_t s) {
  HalfArgs<kMaxSegs> d;
  CombineArgs c;
  const bool fused = k_new != nullptr, bf = quant == PKV_QUANT_BF16;
  int64_t total = 0;
  for (int i = 0; i < n; ++i) {
    HalfSeg &g = d.seg[i];
    g.k = in[i].k;
    g.v = in[i].v;
    g.seq_k = fused ? in[i].seq_k - 1 : in[i].seq_k;
    g.t_new = in[i].seq_k - 1;
    g.nblk = (int)((g.seq_k + kBlk - 1) / kBlk);
    total += g.nblk;
  }
  int slots = 0;
  for (int i = 0; i < n; ++i) {
    HalfSeg &g = d.seg[i];
    int64_t share = total > 0 ? (g.nblk * (int64_t)kHdTargetWGs + total / 2) / total : 1;
    if (share > (g.nblk + 1) / 2) share = (g.nblk + 1) / 2;
    g.nwg = share < 1 ? 1 : (int)share;
    g.wg0 = slots;
    c.wg0[i] = slots;
    slots += g.nwg;
    c.wg1[i] = slots;
  }
  const size_t part_floats = (size_t)slots * 16 * kPartRow, ml_floats = (size_t)slots * 16 * 2;
  const int rc = ws.reserve((part_floats + ml_floats + (size_t)n * 4 * 256) * sizeof(float));
  if (rc) return rc;
  d.rs_t = rs_t;
  d.rs_h = rs_h;
  d.nseg = n;
  d.fused = fused;
  d.sl2 = scale * kLog2e;
  d.q = q;
  d.k_new = k_new;
  d.v_new = v_new;
  d.part = static_cast<float *>(ws.ptr);
  d.ml = reinterpret_cast<float2 *>(d.part + part_floats);
  d.dq = d.part + part_floats + ml_floats;
  const dim3 grid((unsigned)slots), block(kHdThreads);
  if (n == 1) {
    HalfArgs<1> d1;
    d1.rs_t = d.rs_t;
    d1.rs_h = d.rs_h;
    d1.nseg = 1;
    d1.fused = d.fused;
    d1.sl2 = d.sl2;
    d1.q = q;
    d1.k_new = k_new;
    d1.v_new = v_new;
    d1.part = d.part;
    d1.ml = d.ml;
    d1.dq = d.dq;
    d1.seg[0] = d.seg[0];
    if (bf)
      hipLaunchKernelGGL((half_decode_kernel<true, 1>), grid, block, 0, s, d1);
    else
      hipLaunchKernelGGL((half_decode_kernel<false, 1>), grid, block, 0, s, d1);
  } else if (bf) {
    hipLaunchKernelGGL((half_decode_kernel<true, kMaxSegs>), grid, block, 0, s, d);
  } else {
    hipLaunchKernelGGL((half_decode_kernel<false, kMaxSegs>), grid, block, 0, s, d);
  }
  PKV_HIP(hipGetLastError());
  c.part = d.part;
  c.ml = d.ml;
  c.q = q;
  c.dq = fused ? d.dq : nullptr;
  c.out = out;
  c.sl2 = d.sl2;
  return launch_combine(c, n, s);
}

bool half_shape(int quant, int num_heads, int num_kv_heads, int head_dim) {
  return (quant == PKV_QUANT_F16 || quant == PKV_QUANT_BF16) && head_dim == 256 &&
         num_heads == 16 && num_kv_heads == 2;
}
// 16-byte loads from every row
bool half_aligned(const void *k, const void *v, int64_t rs_b, int64_t rs_t, int64_t rs_h) {
  return ((reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) | (uintptr_t)rs_b |
           (uintptr_t)rs_t | (uintptr_t)rs_h) & 15) == 0 && rs_t > 0 && rs_h >= 0 && rs_b >= 0;
}

}  // namespace

int launch_attend_half(const AttnArgs &a, const float *k_new, const float *v_new, uint8_t *kc,
                       uint8_t *vc, int64_t t_new, Workspace &ws, hipStream_t s) {
  if (!half_shape(a.quant, a.num_heads, a.num_kv_heads, a.head_dim) || a.l != 1)
    return PKV_ERR_UNSUPPORTED;
  // decode only: the single query sees every key
  if (a.causal && a.q_offset + 1 < a.seq_k) return PKV_ERR_UNSUPPORTED;
  const bool fused = k_new != nullptr;
  if (fused && (kc != a.k || vc != a.v || t_new != a.seq_k - 1)) return PKV_ERR_UNSUPPORTED;
  if (!half_aligned(a.k, a.v, a.rs.b, a.rs.t, a.rs.h) || !decode_rows_fit(a.seq_k, a.rs.t) ||
      (reinterpret_cast<uintptr_t>(a.q) & 15) != 0)
    return PKV_ERR_UNSUPPORTED;
  if (ws.fixed)
    if (const int rc = generic_plan_fits(a, ws)) return rc;
  for (int b0 = 0; b0 < a.batch; b0 += kMaxSegs) {
    const int nb = a.batch - b0 < kMaxSegs ? a.batch - b0 : kMaxSegs;
    DecodeSegIn in[kMaxSegs];
    for (int i = 0; i < nb; ++i) {
      in[i].k = const_cast<uint8_t *>(a.k) + (int64_t)(b0 + i) * a.rs.b;
      in[i].v = const_cast<uint8_t *>(a.v) + (int64_t)(b0 + i) * a.rs.b;
      in[i].seq_k = a.seq_k;
    }
    const int64_t qo = (int64_t)b0 * 16 * 256, ko = (int64_t)b0 * 2 * 256;
    const int rc = launch_half_segments(a.quant, in, nb, a.q + qo, fused ? k_new + ko : nullptr,
                                        fused ? v_new + ko : nullptr, a.out + qo, a.rs.t, a.rs.h,
                                        a.scale, ws, s);
    if (rc) return rc;
  }
  return PKV_OK;
}

int launch_append_attend_batched_half(int quant, const SeqDesc *seqs, int n, const float *k,
                                      const float *v, const float *q, int num_heads,
                                      int num_kv_heads, int head_dim, float scale, float *out,
                                      Workspace &ws, hipStream_t s) {
  if (!half_shape(quant, num_heads, num_kv_heads, head_dim)) return PKV_ERR_UNSUPPORTED;
  const int64_t rs_t = 2 * 512, rs_h = 512;
  if ((reinterpret_cast<uintptr_t>(q) & 15) != 0) return PKV_ERR_UNSUPPORTED;
  for (int i = 0; i < n; ++i)
    if (seqs[i].len < 1 || !half_aligned(seqs[i].k, seqs[i].v, 0, rs_t, rs_h) ||
        !decode_rows_fit(seqs[i].len, rs_t))
      return PKV_ERR_UNSUPPORTED;
  for (int b0 = 0; b0 < n; b0 += kMaxSegs) {
    const int nb = n - b0 < kMaxSegs ? n - b0 : kMaxSegs;
    DecodeSegIn in[kMaxSegs];
    for (int i = 0; i < nb; ++i) {
      in[i].k = seqs[b0 + i].k;
      in[i].v = seqs[b0 + i].v;
      in[i].seq_k = seqs[b0 + i].len;
    }
    const int64_t qo = (int64_t)b0 * 16 * 256, ko = (int64_t)b0 * 2 * 256;
    const int rc = launch_half_segments(quant, in, nb, q + qo, k + ko, v + ko, out + qo, rs_t, rs_h,
                                        scale, ws, s);
    if (rc) return rc;
  }
  return PKV_OK;
}

}  // namespace pkv
