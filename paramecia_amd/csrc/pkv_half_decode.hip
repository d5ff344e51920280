// MFMA decode attention over F16 and BF16 caches of the Qwen3-Next full-attention shape
// (16 query heads, 2 KV heads, head_dim 256), gfx950.
//
// Role: the CPU SDPA of the reference's float cache (paramecia-model/src/qwen3_next.rs:
// 2492-2605) for a decode step: every query head reads the keys of KV head h / 8, scores
// scaled, clamped to +-100, soft-maxed and applied to V.
//
// Bound: HBM (2048 bytes per cached key) for long caches, the chain of latencies of one
// 32-key block for short ones, so a block's work is split over the workgroup. A workgroup
// of 4 waves owns a range of blocks of one KV head of one segment (a cache's batch row, or
// a sequence). The rows' halves are MFMA operands as they are and go from memory straight
// into registers, a block ahead:
//   QK: wave w takes elements 64 w .. 64 w + 63 of all 32 keys (A: lane (r, g) holds 8
//       elements of key kk(r, t)); the waves' partial scores meet in LDS, one barrier per
//       block, and every wave then runs the same softmax;
//   PV: wave w takes columns e = 64 w + 4 n + j: lane (n, g) reads the 8 bytes of columns
//       4 n .. + 3 of keys 8 g .. 8 g + 7, and pairs of keys become B operands with one
//       v_perm per pair and column.
// Keys are permuted inside a block so that the QK result layout is the PV A layout. The
// new token of a fused step is converted by the first workgroups and joins in the combine
// (pkv_decode_split.hpp) from its rounded rows.
// One layer's step (append, attention, combine), us: 12290 keys 160 before, 12.9 now
// (25.2 MB); 100 keys 7.5, 4096 8.8, 32768 20, 131072 56 (268 MB, 4.8 TB/s). Tried: a wave
// per block and KV head with its merge in LDS (14.4 at 100 keys, 16.0 at 12290: one wave's
// serial work), 384 and 512 slots (14.4 and 15.1 at 12290: the combine reads more).
// Precision: q and the weights p enter as sums of 16-bit parts, accumulated in f32: F16 hi
// and lo (q scaled by a power of two per row, p by 2^11, so that neither part leaves fp16's
// range: 22 bits), BF16 three parts (24 bits). Mean error against 64 bits over 20 to 12000
// keys with scores of standard deviation 0.01 / 1 / 4: 0.24 to 1.1 times the general
// kernel's (12000 keys, 1: F16 1.9e-7 of 5.2e-7).
//
// Infinities and NaN (a float cache stores what it is given; F16 overflows to infinity):
// a split operand times infinity can give inf - inf, so a wave whose scores or sums come
// out non-finite redoes its blocks in plain f32 products (slow_heads), element for element
// what the general kernel (pkv_attn.hip) computes.
#include "pkv_decode_split.hpp"
#include "pkv_half_common.hpp"
#include "pkv_mfma_common.hpp"

namespace pkv {

namespace {

constexpr int kHdWaves = 4, kHdThreads = 64 * kHdWaves;
constexpr int kHdSlots = 256;  // partial slots of a full launch, two workgroups (KV heads) each

struct HalfSeg {
  uint8_t *k, *v;  // rows of token 0, KV head 0
  int64_t seq_k;   // keys attended here (a fused step's new key joins in the combine)
  int64_t t_new;   // row the fused step writes
  int nblk, wg0, nwg;  // its blocks; its first slot, its slots
};
template <int kSegs>
struct HalfArgs {
  int nseg, fused;
  float sl2;    // scale * log2(e)
  float *part;                 // [slot][16][256] in tile order
  float2 *ml;                  // [slot][16]
  float *dq;                   // [nseg][4][256]
  HalfSeg seg[kSegs];
};

// Partial scores of one block: [wave][head][key], rows padded so that the 8 heads' 16-byte
// reads fall on different banks.
constexpr int kScoreStride = 36;
struct HalfSmem {
  __attribute__((aligned(16))) float sc[2][kHdWaves][8][kScoreStride];
  uint32_t bad;
};

// Heads h0 and h0 + 1 of a workgroup's blocks [b0, b1) in f32 products (see the header),
// stored as its partial.
__device__ __forceinline__ void slow_heads(const uint8_t *kbase, const uint8_t *vbase,
                                           int64_t rs_t, int64_t seq_k, int b0, int b1,
                                           const float *q, int h0, float sl2, bool bf, int lane,
                                           float *part, float2 *ml) {
  const int64_t k1 = (int64_t)b1 * kBlk < seq_k ? (int64_t)b1 * kBlk : seq_k;
  float m[2], l[2], acc[2][4];
  half_slow_keys<2>(kbase, vbase, rs_t, (int64_t)b0 * kBlk, k1, q + h0 * 256, sl2, bf, lane, m, l, acc);
#pragma unroll
  for (int x = 0; x < 2; ++x) {
#pragma unroll
    for (int k = 0; k < 4; ++k) part[(h0 + x) * kPartRow + tile_index(4 * lane + k)] = acc[x][k];
    if (lane == 0) ml[h0 + x] = float2{m[x], l[x]};
  }
}

// The leading scalar arguments (segment 0's rows and keys, q, the new rows, rs_t | rs_h <<
// 24, the workgroups) are preloaded into SGPRs, so a one-segment launch's first loads wait
// for no kernel-argument fetch. knew_0 / vnew_0 are q_0 in an attention without an append.
template <bool kBf, int kSegs>
__global__ __launch_bounds__(kHdThreads) void half_decode_kernel(
    const uint8_t *k_0, const uint8_t *v_0, const float *q_0, const float *knew_0,
    const float *vnew_0, uint64_t strides, int seq_k0, int nwg_0, HalfArgs<kSegs> a) {
  __shared__ HalfSmem sm;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slot = (int)blockIdx.x >> 1, kv = (int)blockIdx.x & 1;
  int s = 0;
  if constexpr (kSegs > 1)
    while (s + 1 < a.nseg && a.seg[s + 1].wg0 <= slot) ++s;
  HalfSeg sg;
  if constexpr (kSegs == 1) {
    sg.k = const_cast<uint8_t *>(k_0);
    sg.v = const_cast<uint8_t *>(v_0);
    sg.seq_k = seq_k0;
    sg.nblk = (seq_k0 + kBlk - 1) / kBlk;
    sg.wg0 = 0;
    sg.nwg = nwg_0;
  } else {
    sg = a.seg[s];
  }
  const int64_t rs_h = (int64_t)(strides >> 24);
  // blocks [b0, b1) of the segment
  const int w = slot - sg.wg0, bq = sg.nblk / sg.nwg, br = sg.nblk % sg.nwg;
  const int b0 = w * bq + (w < br ? w : br), b1 = b0 + bq + (w < br ? 1 : 0);
  const uint32_t rs_t = (uint32_t)(strides & 0xFFFFFFu);
  const uint8_t *kbase = sg.k + kv * rs_h, *vbase = sg.v + kv * rs_h;
  const int last = (int)sg.seq_k - 1;  // loads past it read the last row again (masked)
  const uint32_t span = sg.seq_k > 0 ? (uint32_t)last * rs_t + 512u : 0u;
  const __amdgpu_buffer_rsrc_t rk =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(kbase), 0, span, 0x00020000);
  const __amdgpu_buffer_rsrc_t rv =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(vbase), 0, span, 0x00020000);
  u4 kw[2][2];
  uint2 vw[8];
  auto load_k = [&](int b) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int key = b * kBlk + 8 * (n >> 2) + 4 * t + (n & 3);
      const uint32_t off = (uint32_t)(key < last ? key : last) * rs_t + 128u * wave + 16u * g;
#pragma unroll
      for (int st = 0; st < 2; ++st) kw[t][st] = row_load<u4>(rk, off + 64 * st);
    }
  };
  auto load_v = [&](int b) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int key = b * kBlk + 8 * g + k;
      vw[k] = row_load<uint2>(rv, (uint32_t)(key < last ? key : last) * rs_t + 128u * wave + 8u * n);
    }
  };
  const float *qseg = q_0 + ((int64_t)s * 16 + 8 * kv) * 256;
  // q: lane (n, g) holds elements 64 wave + 32 st + 8 g .. + 7 of head n % 8
  float4 qv[2][2];
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int x = 0; x < 2; ++x)
      qv[st][x] = *reinterpret_cast<const float4 *>(qseg + (n & 7) * 256 + 64 * wave + 32 * st + 8 * g + 4 * x);
  // (every workgroup loads a new row's element, so that the load sits in no branch and is
  // waited for where it is used)
  const int new0 = (int)blockIdx.x < 4 * a.nseg ? (int)blockIdx.x : 0;
  float xn = ((new0 & 2) ? vnew_0 : knew_0)[((int64_t)(new0 >> 2) * 2 + (new0 & 1)) * 256 + tid];
  if (b0 < b1) {
    load_k(b0);
    load_v(b0);
  }
  if (tid == 0) sm.bad = 0u;

  // Fused step: row 4 i + 2 p + kv (segment i, K (p = 0) or V) is converted and stored
  if (a.fused) {
    for (int row = blockIdx.x; row < 4 * a.nseg; row += gridDim.x) {
      const int i = row >> 2, p = (row >> 1) & 1, h = row & 1;
      if (row != (int)blockIdx.x) xn = (p ? vnew_0 : knew_0)[((int64_t)i * 2 + h) * 256 + tid];
      const uint16_t y = kBf ? f32_to_bf16(xn) : f32_to_f16(xn);
      const HalfSeg &r = a.seg[kSegs > 1 ? i : 0];
      reinterpret_cast<uint16_t *>((p ? r.v : r.k) + r.t_new * rs_t + h * rs_h)[tid] = y;
      a.dq[(int64_t)row * 256 + tid] = half_value(y, kBf);
    }
  }

  float f = 1.0f, back = 1.0f;  // q enters times f, a partial score leaves times 1 / f
  if constexpr (!kBf) {  // the wave's elements of a row to [2^14, 2^15)
    float mx = 0.0f;
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int x = 0; x < 2; ++x)
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(qv[st][x].x), fabsf(qv[st][x].y)),
                             fmaxf(fabsf(qv[st][x].z), fabsf(qv[st][x].w))));
    mx = xmax32(xmax16(mx));
    int e = (int)(f2u(mx) >> 23) - 127;
    e = e < -100 ? -100 : e > 100 ? 100 : e;
    f = __builtin_ldexpf(1.0f, 14 - e);
    back = __builtin_ldexpf(1.0f, e - 14);
  }
  if (wave & 1) f = -f, back = -back;  // waves 1 and 3 sum negated, as the odd columns do
  u4 qb[2], qb2[2];
#pragma unroll
  for (int st = 0; st < 2; ++st) {
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
  f4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = zero;
  // Scores and the running max stay in q . k units; each exponent is the fma of the score's
  // two summands (rounding a score of tens of log2 units instead cost 2-4 times the error
  // where a few keys dominate, one fma of the rounded sum 1.3 times). F16's factor 2^11 is a product of its own: in the exponent it would
  // round the small ones of the keys that matter.
  constexpr float kUp = kBf ? 1.0f : kPUp;
  const float cs = a.sl2, clamp = kClampL2 / cs, lazy = (kBf ? kBf16Lazy : kF16Lazy) / cs;
  float m_run = -INFINITY, nm = INFINITY, lsum = 0.0f;
  bool bad = false;
  for (int b = b0; b < b1; ++b) {
    // ---- the wave's part of the scores: keys 8 g + 4 t + i, head n % 8 (hi columns n < 8,
    // lo columns n >= 8)
    float(*sc)[8][kScoreStride] = sm.sc[(b - b0) & 1];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f4 c = zero;
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        c = half_mfma<kBf>(kw[t][st], qb[st], c);
        if constexpr (kBf) c = half_mfma<kBf>(kw[t][st], qb2[st], c);
      }
      float4 r;
      r.x = (c[0] + ror8(c[0])) * back;
      r.y = (c[1] + ror8(c[1])) * back;
      r.z = (c[2] + ror8(c[2])) * back;
      r.w = (c[3] + ror8(c[3])) * back;
      if (n < 8) *reinterpret_cast<float4 *>(&sc[wave][n][8 * g + 4 * t]) = r;
    }
    if (b + 1 < b1) load_k(b + 1);
    // (the scores alternate between two buffers: a wave that is a block ahead writes the
    // other one)
    lds_barrier();
    float sc8[8], ca[8], cb[8];  // sc8 = ca + cb, rounded
    {
      float4 pw[kHdWaves][2];
#pragma unroll
      for (int x = 0; x < kHdWaves; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
          pw[x][y] = *reinterpret_cast<const float4 *>(&sc[x][n & 7][8 * g + 4 * y]);
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        ca[4 * y] = pw[0][y].x + pw[1][y].x, cb[4 * y] = pw[2][y].x + pw[3][y].x;
        ca[4 * y + 1] = pw[0][y].y + pw[1][y].y, cb[4 * y + 1] = pw[2][y].y + pw[3][y].y;
        ca[4 * y + 2] = pw[0][y].z + pw[1][y].z, cb[4 * y + 2] = pw[2][y].z + pw[3][y].z;
        ca[4 * y + 3] = pw[0][y].w + pw[1][y].w, cb[4 * y + 3] = pw[2][y].w + pw[3][y].w;
      }
    }
    float big = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      sc8[k] = ca[k] + cb[k];
      big = fmaxf(big, fabsf(sc8[k]));
      bad |= !(fabsf(sc8[k]) < INFINITY);
    }
    if (__any(big > clamp)) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (!(fabsf(sc8[k]) > clamp)) continue;
        sc8[k] = ca[k] = __builtin_amdgcn_fmed3f(sc8[k], -clamp, clamp);
        cb[k] = 0.0f;
      }
    }
    const int nvalid = (int)sg.seq_k - b * kBlk;
    if (nvalid < kBlk) {
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (8 * g + k >= nvalid) sc8[k] = ca[k] = -INFINITY;
    }
    // ---- online softmax (lanes n, n + 16, n + 32, n + 48 hold a head's 32 keys)
    float bm = sc8[0];
#pragma unroll
    for (int k = 1; k < 8; ++k) bm = fmaxf(bm, sc8[k]);
    bm = xmax32(xmax16(bm));
    if (m_run == -INFINITY) {
      m_run = bm;
      nm = -(bm * cs);
    } else if (__any(bm > m_run + lazy)) {
      m_run = fmaxf(m_run, bm);
      const float nm_new = -(m_run * cs);
      const float alpha = __builtin_amdgcn_exp2f(nm_new - nm);
      lsum *= alpha;
      nm = nm_new;
      float ai[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) ai[i] = __shfl(alpha, 4 * (g & 1) + i);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[j][i] *= ai[i];
    }
    float p[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      p[k] = __builtin_amdgcn_exp2f(fmaf(cb[k], cs, fmaf(ca[k], cs, nm))) * kUp;
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
    // ---- PV: tile j, column n: e = 64 wave + 4 n + j (odd tiles negated)
    const u4 An = half_neg(A), A2n = half_neg(A2);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
      uint32_t bw[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        bw[k] = j < 2 ? __builtin_amdgcn_perm(vw[2 * k + 1].x, vw[2 * k].x, sel)
                      : __builtin_amdgcn_perm(vw[2 * k + 1].y, vw[2 * k].y, sel);
      const u4 B = {bw[0], bw[1], bw[2], bw[3]};
      acc[j] = half_mfma<kBf>((j & 1) ? An : A, B, acc[j]);
      if constexpr (kBf) acc[j] = half_mfma<kBf>((j & 1) ? A2n : A2, B, acc[j]);
    }
    if (b + 1 < b1) load_v(b + 1);
  }

  // ---- the partial: rows h and h + 8 summed (lanes 0-31 keep tiles 0 and 1, lanes 32-63
  // tiles 2 and 3), heads 4 (g & 1) + i, in tile order (tile_index of the columns)
  lsum += __shfl_xor(lsum, 16);
  lsum += __shfl_xor(lsum, 32);
  float *part = a.part + ((int64_t)slot * 16 + 8 * kv) * kPartRow;
  float2 *ml = a.ml + (int64_t)slot * 16 + 8 * kv;
  float r[2][4];
#pragma unroll
  for (int y = 0; y < 2; ++y)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      r[y][i] = pair_sum32(acc[y][i], acc[y + 2][i]);
      r[y][i] *= y ? -1.0f / kUp : 1.0f / kUp;
      bad |= !(fabsf(r[y][i]) < INFINITY);
    }
  if (bad) sm.bad = 1u;
  lds_barrier();
  if (sm.bad != 0u) {
    slow_heads(kbase, vbase, rs_t, sg.seq_k, b0, b1, qseg, 2 * wave, a.sl2, kBf, lane, part, ml);
    return;
  }
#pragma unroll
  for (int y = 0; y < 2; ++y) {
    const int at = tile_index(64 * wave + 4 * n + 2 * (g >> 1) + y);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_nontemporal_store(r[y][i], part + (4 * (g & 1) + i) * kPartRow + at);
  }
  if (wave == 0 && lane < 8) ml[n] = float2{-nm, lsum * (1.0f / kUp)};
}

// Plan and launch the decode and the combine over n <= kMaxSegs segments. Every segment
// gets slots in proportion to its blocks, at most one per block and about kHdSlots in all
// (and at least one each).
int launch_half_segments(int quant, const DecodeSegIn *in, int n, const float *q,
                         const float *k_new, const float *v_new, float *out, int64_t rs_t,
                         int64_t rs_h, float scale, Workspace &ws, hipStream_t s) {
  if (!decode_head_stride_fits(rs_h)) return PKV_ERR_UNSUPPORTED;
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
    int64_t share = total > 0 ? (g.nblk * (int64_t)kHdSlots + total / 2) / total : 1;
    if (share > g.nblk) share = g.nblk;
    g.nwg = share < 1 ? 1 : (int)share;
    g.wg0 = slots;
    c.wg0[i] = slots;
    slots += g.nwg;
    c.wg1[i] = slots;
  }
  const size_t part_floats = (size_t)slots * 16 * kPartRow, ml_floats = (size_t)slots * 16 * 2;
  const int rc = ws.reserve((part_floats + ml_floats + (size_t)n * 4 * 256) * sizeof(float));
  if (rc) return rc;
  d.nseg = n;
  d.fused = fused;
  d.sl2 = scale * kLog2e;
  d.part = static_cast<float *>(ws.ptr);
  d.ml = reinterpret_cast<float2 *>(d.part + part_floats);
  d.dq = d.part + part_floats + ml_floats;
  const dim3 grid((unsigned)(2 * slots)), block(kHdThreads);
  const float *kn = fused ? k_new : q, *vn = fused ? v_new : q;
  const uint64_t st = decode_strides(rs_t, rs_h);
  const int seq0 = (int)d.seg[0].seq_k, nwg0 = d.seg[0].nwg;
  if (n == 1) {
    HalfArgs<1> d1;
    d1.nseg = 1;
    d1.fused = d.fused;
    d1.sl2 = d.sl2;
    d1.part = d.part;
    d1.ml = d.ml;
    d1.dq = d.dq;
    d1.seg[0] = d.seg[0];
    if (bf)
      hipLaunchKernelGGL((half_decode_kernel<true, 1>), grid, block, 0, s, d.seg[0].k, d.seg[0].v, q,
                         kn, vn, st, seq0, nwg0, d1);
    else
      hipLaunchKernelGGL((half_decode_kernel<false, 1>), grid, block, 0, s, d.seg[0].k, d.seg[0].v, q,
                         kn, vn, st, seq0, nwg0, d1);
  } else if (bf) {
    hipLaunchKernelGGL((half_decode_kernel<true, kMaxSegs>), grid, block, 0, s, d.seg[0].k,
                       d.seg[0].v, q, kn, vn, st, seq0, nwg0, d);
  } else {
    hipLaunchKernelGGL((half_decode_kernel<false, kMaxSegs>), grid, block, 0, s, d.seg[0].k,
                       d.seg[0].v, q, kn, vn, st, seq0, nwg0, d);
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

}  // namespace

int launch_attend_half(const AttnArgs &a, const float *k_new, const float *v_new, uint8_t *kc,
                       uint8_t *vc, int64_t t_new, Workspace &ws, hipStream_t s) {
  if (!half_shape(a.quant, a.num_heads, a.num_kv_heads, a.head_dim) || a.l != 1)
    return PKV_ERR_UNSUPPORTED;
  // decode only: the single query sees every key
  if (a.causal && a.q_offset + 1 < a.seq_k) return PKV_ERR_UNSUPPORTED;
  const bool fused = k_new != nullptr;
  if (fused && (kc != a.k || vc != a.v || t_new != a.seq_k - 1)) return PKV_ERR_UNSUPPORTED;
  if (!half_scale(a.scale) || !half_aligned(a.k, a.v, a.rs.b, a.rs.t, a.rs.h) || !decode_rows_fit(a.seq_k, a.rs.t) ||
      (reinterpret_cast<uintptr_t>(a.q) & 15) != 0)
    return PKV_ERR_UNSUPPORTED;
  if (ws.fixed)
    if (const int rc = ws.reserve(generic_plan_bytes(a))) return rc;
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
  if ((reinterpret_cast<uintptr_t>(q) & 15) != 0 || !half_scale(scale)) return PKV_ERR_UNSUPPORTED;
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
