// q/k preparation fused into quantize-on-append.
//
// Reference: FullAttention::forward (paramecia-model/src/qwen3_next.rs:2369-2442) runs,
// per layer and step: q_norm on q [b, l, H, d] (candle_nn::ops::rms_norm), k_norm on k
// [b, l, Hkv, d], the transposes to [b, h, l, d], RotaryEmbedding::apply on the first
// n_rot dims (qwen3_next.rs:906-940, candle_nn::rotary_emb::rope, half-split pairs
// (i, i + n_rot/2)) at positions offset + t, and only then append_quantized. Each step
// is its own pass over the rows. Here one launch takes the projection outputs as they
// are ([b, l, h, d]), and finishes each row in one place: a q row (one wave) is normalised
// and rotated into q_out; a K row (one workgroup) is normalised, rotated and encoded into
// the cache; a V row (one workgroup) is encoded. The encoders are the append path's own (Q4K lane quantizer, Q8_0, f16,
// bf16), so the cache bytes equal those of pkv_append on the prepared rows.
//
// Bit-exactness: candle's CPU rms_norm sums x*x sequentially in f32 and computes
// x / sqrt(sum / d + eps) * alpha; rope computes x1*cos - x2*sin and x1*sin + x2*cos
// with every product rounded. Contraction is off for this file, division and sqrt are
// IEEE (hipcc's defaults), and one lane replays the sum in element order.
#pragma clang fp contract(off)

#include "pkv_internal.hpp"
#include "pkv_scalar.hpp"
#include "pkv_q4k_fit.hpp"
#include "pkv_q4k_lanes.hpp"
#include "pkv_prep_common.hpp"

namespace pkv {
namespace {

constexpr int kPrepThreads = 256;  // a K/V row: thread tid owns elements tid, tid + 256
constexpr int kQRowsPerWG = 4;     // q rows of d <= 256: one wave each, 4 elements a lane

struct PrepSmem {
  union {
    struct {
      __attribute__((aligned(16))) float row[512];  // squares, then the normalised row
      float m;
      Q4kScratch q4;
    } kv;
    struct {
      __attribute__((aligned(16))) float row[kQRowsPerWG][256];
      float m[kQRowsPerWG];
    } q;
  };
};

// One wave normalises and rotates a q row of d <= 256 values (lane l: elements 4l..4l+3,
// zero past d), with the same arithmetic as prep_row. row: this wave's 256 LDS floats.
__device__ __forceinline__ void prep_row_wave(float (&x)[4], const PrepElem (&pe)[4], int d,
                                              float eps, int n_rot, float *row, float *m,
                                              int lane) {
#pragma clang fp contract(off)
  *reinterpret_cast<float4 *>(row + 4 * lane) =
      float4{x[0] * x[0], x[1] * x[1], x[2] * x[2], x[3] * x[3]};
  __builtin_amdgcn_wave_barrier();
  if (lane == 0) {
    float sum2 = -0.0f;
    const float4 *r4 = reinterpret_cast<const float4 *>(row);
    int e = 0;
    for (; e + 4 <= d; e += 4) {
      const float4 t = r4[e >> 2];
      sum2 += t.x;
      sum2 += t.y;
      sum2 += t.z;
      sum2 += t.w;
    }
    for (; e < d; ++e) sum2 += row[e];
    *m = __builtin_sqrtf(sum2 / (float)d + eps);
  }
  __builtin_amdgcn_wave_barrier();
  const float mm = *m;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (4 * lane + i < d) x[i] = x[i] / mm * pe[i].alpha;
  if (n_rot == 0) return;
  *reinterpret_cast<float4 *>(row + 4 * lane) = float4{x[0], x[1], x[2], x[3]};
  __builtin_amdgcn_wave_barrier();
  const int half = n_rot >> 1;
  float r[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = 4 * lane + i;
    if (e >= n_rot)
      r[i] = x[i];
    else if (e < half)
      r[i] = x[i] * pe[i].c - row[e + half] * pe[i].s;
    else
      r[i] = row[e - half] * pe[i].s + x[i] * pe[i].c;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = r[i];
}

// Q8_0 (BlockQ8_0::from_float) of element e of a row, 32 lanes per block: the maximum
// of |x| over the block is exact in any order (NaN dropped, as f32::max does).
__device__ __forceinline__ void q8_encode(float x, int e, uint8_t *row) {
  const int32_t key = (x != x) ? 0 : (int32_t)(f2u(x) & 0x7FFFFFFFu);
  const int32_t kmax = halfwave_allreduce(key, [](int32_t p, int32_t q) { return p > q ? p : q; });
  const float amax = u2f((uint32_t)kmax);
  const float d = amax / 127.0f;
  const float id = (d != 0.0f) ? 1.0f / d : 0.0f;
  uint8_t *blk = row + (e >> 5) * 34;
  blk[2 + (e & 31)] = (uint8_t)rs_as_i8(__builtin_roundf(x * id));
  if ((e & 31) == 0) *reinterpret_cast<uint16_t *>(blk) = f32_to_f16(d);
}

// Workgroups [0, q_wgs) prepare q rows (kQRowsPerWG per workgroup when d <= 256, else
// one), then one workgroup per K row, then one per V row. Every global load of a row
// (x, alpha, cos / sin) is issued before the first barrier.
__global__ __launch_bounds__(kPrepThreads) void prep_append_kernel(PrepArgs a, int64_t q_wgs) {
  __shared__ PrepSmem S;
  const int tid = threadIdx.x;
  const int64_t r = blockIdx.x;
  const int d = a.head_dim, n_rot = a.n_rot, half = n_rot >> 1;
  const bool q_by_wave = d <= 256;
  if (r < q_wgs && q_by_wave) {
    const int lane = tid & 63, w = tid >> 6;
    const int64_t i = r * kQRowsPerWG + w;
    if (i >= a.q_rows) return;  // no workgroup barrier on this path
    const int64_t t = (i / a.num_heads) % a.l;
    const int64_t pos = a.t0 + t;
    const float *src = a.q + i * d;
    float x[4];
    PrepElem pe[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int e = 4 * lane + k;
      x[k] = e < d ? src[e] : 0.0f;
      pe[k] = load_prep_elem(a.q_alpha, a.cos_tab + pos * half, a.sin_tab + pos * half, e, d,
                             n_rot);
    }
    prep_row_wave(x, pe, d, a.eps, n_rot, S.q.row[w], &S.q.m[w], lane);
    float *o = a.q_out + i * d;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (4 * lane + k < d) o[4 * lane + k] = x[k];
    return;
  }
  // one row per workgroup from here on
  int kind;  // 0 q (d > 256), 1 K, 2 V
  int64_t i;
  if (r < q_wgs) {
    kind = 0;
    i = r;
  } else if (r < q_wgs + a.kv_rows) {
    kind = 1;
    i = r - q_wgs;
  } else {
    kind = 2;
    i = r - q_wgs - a.kv_rows;
  }
  const int heads = kind == 0 ? a.num_heads : a.kv_heads;
  const int h = (int)(i % heads);
  const int64_t bt = i / heads;  // b * l + t
  const int64_t t = bt % a.l;
  const int b = (int)(bt / a.l);
  const int64_t pos = a.t0 + t;
  const float *src = (kind == 0 ? a.q : kind == 1 ? a.k : a.v) + i * d;
  float x[2] = {tid < d ? src[tid] : 0.0f, tid + 256 < d ? src[tid + 256] : 0.0f};
  if (kind != 2) {
    const float *al = kind == 0 ? a.q_alpha : a.k_alpha;
    const PrepElem pe[2] = {
        load_prep_elem(al, a.cos_tab + pos * half, a.sin_tab + pos * half, tid, d, n_rot),
        load_prep_elem(al, a.cos_tab + pos * half, a.sin_tab + pos * half, tid + 256, d, n_rot)};
    Q4kWorkgroupBarrier bar;
    prep_row<2>(x, pe, d, a.eps, n_rot, S.kv.row, &S.kv.m, tid, bar);
  }
  if (kind == 0) {
    float *o = a.q_out + i * d;
    if (tid < d) o[tid] = x[0];
    if (tid + 256 < d) o[tid + 256] = x[1];
    return;
  }
  uint8_t *row = (kind == 1 ? a.kc : a.vc) + (((a.t0 + t) * a.batch + b) * a.kv_heads + h) * a.bpr;
  if (a.quant == PKV_QUANT_Q4K) {
    q4k_quantize_superblock_lanes(x[0], row, &S.kv.q4, tid);
    if (a.padded > 256) q4k_quantize_superblock_lanes(x[1], row + 144, &S.kv.q4, tid);
  } else if (a.quant == PKV_QUANT_Q8_0) {
    if (tid < a.padded) q8_encode(x[0], tid, row);
    if (tid + 256 < a.padded) q8_encode(x[1], tid + 256, row);
  } else {
    uint16_t *dst = reinterpret_cast<uint16_t *>(row);
    const bool bf = a.quant == PKV_QUANT_BF16;
    if (tid < a.padded) dst[tid] = bf ? f32_to_bf16(x[0]) : f32_to_f16(x[0]);
    if (tid + 256 < a.padded) dst[tid + 256] = bf ? f32_to_bf16(x[1]) : f32_to_f16(x[1]);
  }
}

// ---- many rows (head_dim 256): tiles of rows per workgroup
//
// The row kernel above has one lane add a row's 256 squares in order while the other 63
// (a K row: 255) wait, and quantizes a K or V row as one latency chain: 136 us for 4001
// tokens of Q4K, of which the bytes (147 MB) take about 30 at the copy rate. Here a workgroup takes a tile of rows
// of one kind; the squares of the tile go to LDS and lane r adds those of row r, so the
// ordered sums of all its rows run side by side; the normalised rows are quantized with 8
// kL lanes per row, as pkv_append does (kL from the row count, by the same limits).
// 4001 tokens: 136 -> 42 us Q4K, 66 -> 37 us Q8_0 and F16.
// Rows (q, K and V) from which the tiles are used, and superblocks up to which a K or V
// superblock takes 4 lanes per sub-block (2 above). Model shape, us, rows kernel / tiles:
// Q4K 1 token 7.8 / 7.9, 5 tokens 8.0 / 7.6, 512 25.1 / 10.3; Q8_0 256 tokens 7.6 / 10.3,
// 512 12.4 / 11.0; F16 512 11.7 / 10.9. 4 lanes against 2: 512 tokens 10.4 / 12.9, 1024
// tokens 17.2 / 15.1.
constexpr int64_t kTileMinRowsQ4K = 40, kTileMinRowsOther = 10240, kFit4Blocks = 2048;
constexpr int kTileRows = 16;   // rows of a tile (K and V of few rows: 8)
constexpr int kTileStride = 260;  // floats per LDS row: b128 reads of 8 rows on 32 banks

// Normalise and rotate the kN rows a wave holds in x (lane l: elements 4 l .. 4 l + 3 of row
// r0 + i), with the arithmetic of prep_row. Every wave of the workgroup calls it.
template <int kN>
__device__ __forceinline__ void prep_tile(float4 (&x)[kN], float (*rows)[kTileStride], float *m,
                                          int r0, int nrows, int tid, float4 alpha, float eps,
                                          int n_rot, const float *cos_tab, const float *sin_tab,
                                          const int64_t (&pos)[kN]) {
#pragma clang fp contract(off)
  const int lane = tid & 63, half = n_rot >> 1;
  // the rotation's cos and sin, loaded ahead of the sums: elements 4 lane .. + 3
  const bool rot = 4 * lane < n_rot;
  float cs[kN][4], sn[kN][4];
#pragma unroll
  for (int i = 0; i < kN; ++i)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int e = 4 * lane + k, j = e < half ? e : e - half;
      const bool in = rot && e < n_rot;
      cs[i][k] = in ? cos_tab[pos[i] * half + j] : 1.0f;
      sn[i][k] = in ? sin_tab[pos[i] * half + j] : 0.0f;
    }
#pragma unroll
  for (int i = 0; i < kN; ++i)
    *reinterpret_cast<float4 *>(&rows[r0 + i][4 * lane]) =
        float4{x[i].x * x[i].x, x[i].y * x[i].y, x[i].z * x[i].z, x[i].w * x[i].w};
  __syncthreads();
  if (tid < nrows) {
    float sum2 = -0.0f;
#pragma unroll 16
    for (int e = 0; e < 64; ++e) {
      const float4 t = *reinterpret_cast<const float4 *>(&rows[tid][4 * e]);
      sum2 += t.x;
      sum2 += t.y;
      sum2 += t.z;
      sum2 += t.w;
    }
    m[tid] = __builtin_sqrtf(sum2 / 256.0f + eps);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kN; ++i) {
    const float mm = m[r0 + i];
    x[i].x = x[i].x / mm * alpha.x;
    x[i].y = x[i].y / mm * alpha.y;
    x[i].z = x[i].z / mm * alpha.z;
    x[i].w = x[i].w / mm * alpha.w;
  }
  if (n_rot == 0) return;
  // the rotated elements through the wave's own LDS rows
#pragma unroll
  for (int i = 0; i < kN; ++i)
    if (rot) *reinterpret_cast<float4 *>(&rows[r0 + i][4 * lane]) = x[i];
  __builtin_amdgcn_wave_barrier();
  if (rot) {
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const float *row = rows[r0 + i];
      float v[4] = {x[i].x, x[i].y, x[i].z, x[i].w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int e = 4 * lane + k;
        if (e < half)
          v[k] = v[k] * cs[i][k] - row[e + half] * sn[i][k];
        else if (e < n_rot)
          v[k] = row[e - half] * sn[i][k] + v[k] * cs[i][k];
      }
      x[i] = float4{v[0], v[1], v[2], v[3]};
    }
  }
  __builtin_amdgcn_wave_barrier();
}

// Positions of rows r .. r + kN - 1 of a [batch, l, heads] order: two divisions, then steps
// (a 64-bit division per row took longer than the rest of a tile).
template <int kN>
__device__ __forceinline__ void tile_pos(uint32_t r, uint32_t heads, uint32_t l, int64_t t0,
                                         int64_t (&pos)[kN]) {
  uint32_t bt = r / heads, h = r - bt * heads, t = bt % l;
#pragma unroll
  for (int i = 0; i < kN; ++i) {
    pos[i] = t0 + t;
    if (++h == heads) {
      h = 0;
      t = t + 1 == l ? 0 : t + 1;
    }
  }
}

enum { kTileQ4K, kTileQ8, kTileHalf };

// Workgroups [0, kv_wgs) take K tiles, [kv_wgs, 2 kv_wgs) V tiles (the quantizers are the
// long ones), the rest q tiles.
template <int kFmt, int kL>
__global__ __launch_bounds__(256) void prep_tiles_kernel(PrepArgs a, uint32_t kv_wgs) {
#pragma clang fp contract(off)
  __shared__ __attribute__((aligned(16))) float rows[kTileRows][kTileStride];
  __shared__ float m[kTileRows];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t wg = blockIdx.x;
  if (wg >= 2 * kv_wgs) {
    constexpr int kN = kTileRows / 4;
    const int64_t base = (int64_t)(wg - 2 * kv_wgs) * kTileRows;
    const int r0 = kN * wave;
    float4 x[kN];
    int64_t pos[kN];
#pragma unroll
    for (int i = 0; i < kN; ++i) {  // rows past the last read it again and are not stored
      int64_t r = base + r0 + i;
      r = r < a.q_rows ? r : a.q_rows - 1;
      x[i] = reinterpret_cast<const float4 *>(a.q + r * 256)[lane];
    }
    tile_pos<kN>((uint32_t)(base + r0), (uint32_t)a.num_heads, (uint32_t)a.l, a.t0, pos);
    prep_tile<kN>(x, rows, m, r0, kTileRows, tid, reinterpret_cast<const float4 *>(a.q_alpha)[lane],
                  a.eps, a.n_rot, a.cos_tab, a.sin_tab, pos);
#pragma unroll
    for (int i = 0; i < kN; ++i)
      if (base + r0 + i < a.q_rows)
        reinterpret_cast<float4 *>(a.q_out + (base + r0 + i) * 256)[lane] = x[i];
    return;
  }
  constexpr int kR = kFmt == kTileQ4K && kL == 4 ? 8 : kTileRows, kN = kR / 4;  // of the tile, per wave
  const bool is_v = wg >= kv_wgs;
  const int64_t base = (int64_t)(is_v ? wg - kv_wgs : wg) * kR;
  const float *src = is_v ? a.v : a.k;
  const int r0 = kN * wave;
  float4 x[kN];
  int64_t pos[kN];
#pragma unroll
  for (int i = 0; i < kN; ++i) {
    int64_t r = base + r0 + i;
    r = r < a.kv_rows ? r : a.kv_rows - 1;
    x[i] = reinterpret_cast<const float4 *>(src + r * 256)[lane];
  }
  tile_pos<kN>((uint32_t)(base + r0), (uint32_t)a.kv_heads, (uint32_t)a.l, a.t0, pos);
  if (!is_v)
    prep_tile<kN>(x, rows, m, r0, kR, tid, reinterpret_cast<const float4 *>(a.k_alpha)[lane], a.eps,
                  a.n_rot, a.cos_tab, a.sin_tab, pos);
  // destination row of source row r = (b * l + t) * kv_heads + h
  auto dst_row = [&](int64_t row) {
    const uint32_t r = (uint32_t)row, hs = (uint32_t)a.kv_heads, l = (uint32_t)a.l;
    const uint32_t bt = r / hs, b = bt / l, t = bt - b * l;
    return (is_v ? a.vc : a.kc) + (((a.t0 + t) * a.batch + b) * a.kv_heads + (r - bt * hs)) * a.bpr;
  };
  if constexpr (kFmt == kTileHalf) {
    const bool bf = a.quant == PKV_QUANT_BF16;
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const float v[4] = {x[i].x, x[i].y, x[i].z, x[i].w};
      uint16_t y[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) y[k] = bf ? f32_to_bf16(v[k]) : f32_to_f16(v[k]);
      if (base + r0 + i < a.kv_rows)
        reinterpret_cast<uint2 *>(dst_row(base + r0 + i))[lane] =
            uint2{(uint32_t)y[0] | ((uint32_t)y[1] << 16), (uint32_t)y[2] | ((uint32_t)y[3] << 16)};
    }
  } else {
  // the quantizers: 8 kL lanes per row, each with 32 / kL elements in order
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kN; ++i) *reinterpret_cast<float4 *>(&rows[r0 + i][4 * lane]) = x[i];
  __syncthreads();
  constexpr int E = 32 / kL;
  // (Q8_0: the threads past the tile's blocks leave; no barrier follows)
  const int rr = tid / (8 * kL), r = tid & (8 * kL - 1);
  if (rr >= kR) return;
  float y[E];
#pragma unroll
  for (int i = 0; i < E / 4; ++i) {
    const float4 t = *reinterpret_cast<const float4 *>(&rows[rr][E * r + 4 * i]);
    y[4 * i] = t.x;
    y[4 * i + 1] = t.y;
    y[4 * i + 2] = t.z;
    y[4 * i + 3] = t.w;
  }
  const bool live = base + rr < a.kv_rows;
  if constexpr (kFmt == kTileQ4K) {
    q4k_quantize_group<kL>(y, r, [&] { return dst_row(base + rr); }, live);
  } else {  // one lane per block
    uint8_t *dst = dst_row(live ? base + rr : a.kv_rows - 1);
    static_assert(kL == 1, "Q8_0: one lane per block");
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; ++i) amax = fmax_rs(amax, __builtin_fabsf(y[i]));
    const float d = amax / 127.0f;
    const float id = (d != 0.0f) ? 1.0f / d : 0.0f;
    uint16_t w[17];
    w[0] = f32_to_f16(d);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      w[1 + i] = (uint16_t)((uint32_t)(uint8_t)rs_as_i8(__builtin_roundf(y[2 * i] * id)) |
                            ((uint32_t)(uint8_t)rs_as_i8(__builtin_roundf(y[2 * i + 1] * id)) << 8));
    if (live) {
      uint16_t *o = reinterpret_cast<uint16_t *>(dst + 34 * r);
#pragma unroll
      for (int i = 0; i < 17; ++i) o[i] = w[i];
    }
  }
  }
}

}  // namespace

int launch_prep_append(const PrepArgs &a, hipStream_t s) {
  if (a.head_dim > 512 || a.padded > 512) return set_error(PKV_ERR_UNSUPPORTED, "head_dim > 512");
  const int64_t q_wgs =
      a.head_dim <= 256 ? (a.q_rows + kQRowsPerWG - 1) / kQRowsPerWG : a.q_rows;
  const int64_t grid = q_wgs + 2 * a.kv_rows;
  if (grid == 0) return PKV_OK;
  if (grid >= (1ll << 31)) return set_error(PKV_ERR_ARG, "too many rows in one append");
  // Tiles where the rows are many and the loads may be 16 bytes wide, four elements a lane.
  const uintptr_t ptrs = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.q_out) |
                         reinterpret_cast<uintptr_t>(a.k) | reinterpret_cast<uintptr_t>(a.v) |
                         reinterpret_cast<uintptr_t>(a.q_alpha) |
                         reinterpret_cast<uintptr_t>(a.k_alpha);
  const bool q4 = a.quant == PKV_QUANT_Q4K;
  if (a.head_dim == 256 && (ptrs & 15) == 0 && a.kv_rows > 0 && a.q_rows < (1ll << 31) &&
      a.q_rows + 2 * a.kv_rows >= (q4 ? kTileMinRowsQ4K : kTileMinRowsOther)) {
    const int kl = !q4 ? 1 : a.kv_rows * 2 <= kFit4Blocks ? 4 : 2;
    const int64_t per = kl == 4 ? 8 : kTileRows, kv_wgs = (a.kv_rows + per - 1) / per;
    const dim3 g((unsigned)(2 * kv_wgs + (a.q_rows + kTileRows - 1) / kTileRows)), t(256);
    const uint32_t kw = (uint32_t)kv_wgs;
    if (q4 && kl == 4)
      hipLaunchKernelGGL((prep_tiles_kernel<kTileQ4K, 4>), g, t, 0, s, a, kw);
    else if (q4)
      hipLaunchKernelGGL((prep_tiles_kernel<kTileQ4K, 2>), g, t, 0, s, a, kw);
    else if (a.quant == PKV_QUANT_Q8_0)
      hipLaunchKernelGGL((prep_tiles_kernel<kTileQ8, 1>), g, t, 0, s, a, kw);
    else
      hipLaunchKernelGGL((prep_tiles_kernel<kTileHalf, 1>), g, t, 0, s, a, kw);
    PKV_HIP(hipGetLastError());
    return PKV_OK;
  }
  hipLaunchKernelGGL(prep_append_kernel, dim3((unsigned)grid), dim3(kPrepThreads), 0, s, a,
                     q_wgs);
  PKV_HIP(hipGetLastError());
  return PKV_OK;
}

}  // namespace pkv
