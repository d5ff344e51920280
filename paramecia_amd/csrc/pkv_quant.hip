// Quantize-on-append and dequantize kernels for the packed KV rows.
//
// Reference: PreallocatedQuantizedKvCache::append_quantized
// (paramecia-model/src/qwen3_next.rs:431-509) quantizes the new [b, h, n, d] K/V on
// the CPU with candle's QTensor::quantize and memcpy's the rows at
// seq_len*b*h*bytes_per_row; get_kv (qwen3_next.rs:520-575) dequantizes them.
// Here both run on the GPU, writing/reading the same seq-major rows in HBM.
//
// Bit-exactness: every a*b+c below must round twice like the Rust code, so
// contraction is off for this whole file, divisions are IEEE (hipcc's default), and
// each Q4K sub-block's sums run sequentially in one lane.
#pragma clang fp contract(off)

#include "pkv_internal.hpp"
#include "pkv_scalar.hpp"
#include "pkv_q4k_fit.hpp"
#include "pkv_q4k_lanes.hpp"

namespace pkv {
namespace {

struct AppendArgs {
  const float *src[2];  // k, v: [batch, heads, n, head_dim]
  uint8_t *dst[2];      // K, V row buffers (paged: the pool's K and V page planes)
  int batch, heads, head_dim, padded;
  int64_t n, t0;
  int64_t bpr;
  // Paged rows (page_tab non-null): token t lives in page page_tab[t >> page_lg], row
  // t & (2^page_lg - 1) of that page, each page page_bytes long in each plane
  const int32_t *page_tab;
  int page_lg;
  int64_t page_bytes;
  // One token into each of `batch` paged sequences (row_mode): row (b, h) at byte
  // row_off[b] + h * bpr of each plane
  int row_mode;
  int64_t row_off[kAppendSeqs];
};

// Source element e (< padded) of new row (t, b, h); zero padding past head_dim.
__device__ __forceinline__ float load_elem(const float *src, const AppendArgs &a, int64_t t,
                                           int b, int h, int e) {
  if (e >= a.head_dim) return 0.0f;
  return src[(((int64_t)b * a.heads + h) * a.n + t) * a.head_dim + e];
}

__device__ __forceinline__ int64_t dst_row(const AppendArgs &a, int64_t t, int b, int h) {
  return ((a.t0 + t) * a.batch + b) * a.heads + h;
}
// The destination row of new token t (batch row b, head h) in plane p (K 0, V 1).
__device__ __forceinline__ uint8_t *row_ptr(const AppendArgs &a, int p, int64_t t, int b, int h) {
  if (a.row_mode) return a.dst[p] + a.row_off[b] + (int64_t)h * a.bpr;
  if (a.page_tab != nullptr) {
    const int64_t tok = a.t0 + t, in_page = tok & ((int64_t(1) << a.page_lg) - 1);
    const int64_t pg = a.page_tab[tok >> a.page_lg];
    return a.dst[p] + pg * a.page_bytes + ((in_page * a.batch + b) * a.heads + h) * a.bpr;
  }
  return a.dst[p] + dst_row(a, t, b, h) * a.bpr;
}

// One group of 8 kL lanes per superblock (q4k_quantize_group), every superblock of K, then
// of V.
template <int kL>
__global__ __launch_bounds__(256) void q4k_append_kernel(AppendArgs a, int64_t units_per_tensor,
                                                         int nsb) {
  constexpr int E = 32 / kL;
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t unit = gid / (8 * kL);
  const int r = (int)(gid & (8 * kL - 1));
  const int j = r / kL, s = r & (kL - 1);
  const int64_t total = 2 * units_per_tensor;
  const bool active = unit < total;
  if (!active) unit = total - 1;  // compute redundantly, store nothing
  const int p = (int)(unit / units_per_tensor);
  int64_t u = unit % units_per_tensor;
  const int sb = (int)(u % nsb);
  u /= nsb;
  const int h = (int)(u % a.heads);
  u /= a.heads;
  const int b = (int)(u % a.batch);
  const int64_t t = u / a.batch;

  float x[E];
  const int e0 = sb * 256 + 32 * j + s * E;
  const float *src = a.src[p];
  if ((a.head_dim & 3) == 0 && e0 + E <= a.head_dim) {
    const float4 *s4 = reinterpret_cast<const float4 *>(
        src + (((int64_t)b * a.heads + h) * a.n + t) * a.head_dim + e0);
#pragma unroll
    for (int i = 0; i < E / 4; ++i) {
      float4 f = s4[i];
      x[4 * i] = f.x;
      x[4 * i + 1] = f.y;
      x[4 * i + 2] = f.z;
      x[4 * i + 3] = f.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < E; ++i) x[i] = load_elem(src, a, t, b, h, e0 + i);
  }

  q4k_quantize_group<kL>(x, r, row_ptr(a, p, t, b, h) + (int64_t)sb * 144, active);
}

// One workgroup per (tensor, token, batch, head, superblock); for appends of a few rows.
__global__ __launch_bounds__(256) void q4k_append_small_kernel(AppendArgs a, int nsb) {
  __shared__ Q4kScratch scr;
  int64_t u = blockIdx.x;
  const int sb = (int)(u % nsb);
  u /= nsb;
  const int h = (int)(u % a.heads);
  u /= a.heads;
  const int b = (int)(u % a.batch);
  u /= a.batch;
  const int64_t t = u % a.n;
  const int p = (int)(u / a.n);
  const float x = load_elem(a.src[p], a, t, b, h, sb * 256 + (int)threadIdx.x);
  uint8_t *blk = row_ptr(a, p, t, b, h) + (int64_t)sb * 144;
  q4k_quantize_superblock_lanes(x, blk, &scr, (int)threadIdx.x);
}

// Q8_0 (BlockQ8_0::from_float): one lane per 32-element block.
__global__ __launch_bounds__(256) void q8_0_append_kernel(AppendArgs a, int64_t units_per_tensor,
                                                          int nblk) {
  const int64_t unit = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (unit >= 2 * units_per_tensor) return;
  const int p = (int)(unit / units_per_tensor);
  int64_t u = unit % units_per_tensor;
  const int blk = (int)(u % nblk);
  u /= nblk;
  const int h = (int)(u % a.heads);
  u /= a.heads;
  const int b = (int)(u % a.batch);
  const int64_t t = u / a.batch;
  float x[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) x[i] = load_elem(a.src[p], a, t, b, h, blk * 32 + i);
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 32; ++i) amax = fmax_rs(amax, __builtin_fabsf(x[i]));
  const float d = amax / 127.0f;
  const float id = (d != 0.0f) ? 1.0f / d : 0.0f;
  uint16_t w[17];
  w[0] = f32_to_f16(d);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    uint32_t q0 = (uint8_t)rs_as_i8(__builtin_roundf(x[2 * i] * id));
    uint32_t q1 = (uint8_t)rs_as_i8(__builtin_roundf(x[2 * i + 1] * id));
    w[1 + i] = (uint16_t)(q0 | (q1 << 8));
  }
  uint16_t *dst =
      reinterpret_cast<uint16_t *>(row_ptr(a, p, t, b, h) + (int64_t)blk * 34);
#pragma unroll
  for (int i = 0; i < 17; ++i) dst[i] = w[i];
}

// F16 / BF16 rows: element-wise round-to-nearest-even conversion.
template <bool BF>
__global__ __launch_bounds__(256) void half_append_kernel(AppendArgs a, int64_t elems_per_tensor) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 2 * elems_per_tensor) return;
  const int p = (int)(i / elems_per_tensor);
  int64_t u = i % elems_per_tensor;
  const int e = (int)(u % a.padded);
  u /= a.padded;
  const int h = (int)(u % a.heads);
  u /= a.heads;
  const int b = (int)(u % a.batch);
  const int64_t t = u / a.batch;
  const float x = load_elem(a.src[p], a, t, b, h, e);
  uint16_t *dst = reinterpret_cast<uint16_t *>(row_ptr(a, p, t, b, h));
  dst[e] = BF ? f32_to_bf16(x) : f32_to_f16(x);
}

__global__ __launch_bounds__(256) void dequant_kernel(int quant, const uint8_t *kc,
                                                      const uint8_t *vc, float *ko, float *vo,
                                                      int batch, int heads, int head_dim,
                                                      int64_t S, int64_t bpr) {
  const int64_t per = (int64_t)batch * heads * S * head_dim;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 2 * per) return;
  const int p = (int)(i / per);
  int64_t u = i % per;  // index into [b, h, S, d]
  const int e = (int)(u % head_dim);
  u /= head_dim;
  const int64_t t = u % S;
  u /= S;
  const int h = (int)(u % heads);
  const int b = (int)(u / heads);
  const int64_t r = (t * batch + b) * heads + h;
  const uint8_t *row = (p ? vc : kc) + r * bpr;
  (p ? vo : ko)[i % per] = decode_elem(quant, row, e);
}

}  // namespace

static int launch_append_args(int quant, AppendArgs &a, hipStream_t s);

int launch_append(int quant, const float *k, const float *v, uint8_t *kc, uint8_t *vc,
                  int batch, int heads, int head_dim, int64_t n, int64_t t0, hipStream_t s) {
  if (n == 0) return PKV_OK;
  AppendArgs a;
  a.src[0] = k;
  a.src[1] = v;
  a.dst[0] = kc;
  a.dst[1] = vc;
  a.batch = batch;
  a.heads = heads;
  a.head_dim = head_dim;
  a.padded = padded_dim(quant, head_dim);
  a.n = n;
  a.t0 = t0;
  a.bpr = (int64_t)row_bytes(quant, head_dim);
  a.page_tab = nullptr;
  a.page_lg = 0;
  a.page_bytes = 0;
  a.row_mode = 0;
  return launch_append_args(quant, a, s);
}

int launch_append_paged(int quant, const float *k, const float *v, uint8_t *kpool,
                        uint8_t *vpool, const int32_t *page_tab, int page_lg,
                        int64_t page_bytes, int heads, int head_dim, int64_t n, int64_t t0,
                        hipStream_t s) {
  if (n == 0) return PKV_OK;
  AppendArgs a;
  a.src[0] = k;
  a.src[1] = v;
  a.dst[0] = kpool;
  a.dst[1] = vpool;
  a.batch = 1;
  a.heads = heads;
  a.head_dim = head_dim;
  a.padded = padded_dim(quant, head_dim);
  a.n = n;
  a.t0 = t0;
  a.bpr = (int64_t)row_bytes(quant, head_dim);
  a.page_tab = page_tab;
  a.page_lg = page_lg;
  a.page_bytes = page_bytes;
  a.row_mode = 0;
  return launch_append_args(quant, a, s);
}

int launch_append_rows(int quant, const float *k, const float *v, uint8_t *kpool, uint8_t *vpool,
                       const int64_t *row_off, int n, int heads, int head_dim, hipStream_t s) {
  if (n <= 0) return PKV_OK;
  if (n > kAppendSeqs) return set_error(PKV_ERR_ARG, "too many rows for one append launch");
  AppendArgs a;
  a.src[0] = k;
  a.src[1] = v;
  a.dst[0] = kpool;
  a.dst[1] = vpool;
  a.batch = n;
  a.heads = heads;
  a.head_dim = head_dim;
  a.padded = padded_dim(quant, head_dim);
  a.n = 1;
  a.t0 = 0;
  a.bpr = (int64_t)row_bytes(quant, head_dim);
  a.page_tab = nullptr;
  a.page_lg = 0;
  a.page_bytes = 0;
  a.row_mode = 1;
  for (int i = 0; i < n; ++i) a.row_off[i] = row_off[i];
  return launch_append_args(quant, a, s);
}

// Q4K superblocks (K and V) up to which the throughput kernel runs 4, then 2, lanes per
// sub-block (1 above)
constexpr int64_t kQ4kAppendLanes4Max = 2048, kQ4kAppendLanes2Max = 8192;

static int launch_append_args(int quant, AppendArgs &a, hipStream_t s) {
  const int batch = a.batch, heads = a.heads;
  const int64_t n = a.n;
  const int64_t rows = n * batch * heads;
  if (quant == PKV_QUANT_Q4K && rows * (a.padded / 256) * 2 <= 1024) {
    // few superblocks: latency-bound, one workgroup each
    const int nsb = a.padded / 256;
    hipLaunchKernelGGL(q4k_append_small_kernel, dim3((unsigned)(2 * rows * nsb)), dim3(256), 0,
                       s, a, nsb);
  } else if (quant == PKV_QUANT_Q4K) {
    // 8 kL lanes per superblock: split each sub-block's fit over more lanes while the
    // append has too few superblocks to give every SIMD a wave
    const int nsb = a.padded / 256;
    const int64_t units = rows * nsb;
    const int kl = 2 * units <= kQ4kAppendLanes4Max ? 4 : (2 * units <= kQ4kAppendLanes2Max ? 2 : 1);
    const int64_t threads = 2 * units * 8 * kl;
    const dim3 grid((unsigned)((threads + 255) / 256));
    if (kl == 4)
      hipLaunchKernelGGL(q4k_append_kernel<4>, grid, dim3(256), 0, s, a, units, nsb);
    else if (kl == 2)
      hipLaunchKernelGGL(q4k_append_kernel<2>, grid, dim3(256), 0, s, a, units, nsb);
    else
      hipLaunchKernelGGL(q4k_append_kernel<1>, grid, dim3(256), 0, s, a, units, nsb);
  } else if (quant == PKV_QUANT_Q8_0) {
    const int nblk = a.padded / 32;
    const int64_t units = rows * nblk;
    hipLaunchKernelGGL(q8_0_append_kernel, dim3((unsigned)((2 * units + 255) / 256)), dim3(256),
                       0, s, a, units, nblk);
  } else {
    const int64_t elems = rows * a.padded;
    if (quant == PKV_QUANT_BF16)
      hipLaunchKernelGGL(half_append_kernel<true>, dim3((unsigned)((2 * elems + 255) / 256)),
                         dim3(256), 0, s, a, elems);
    else
      hipLaunchKernelGGL(half_append_kernel<false>, dim3((unsigned)((2 * elems + 255) / 256)),
                         dim3(256), 0, s, a, elems);
  }
  PKV_HIP(hipGetLastError());
  return PKV_OK;
}

int launch_dequant(int quant, const uint8_t *kc, const uint8_t *vc, float *ko, float *vo,
                   int batch, int heads, int head_dim, int64_t S, hipStream_t s) {
  const int64_t total = 2 * (int64_t)batch * heads * S * head_dim;
  if (total == 0) return PKV_OK;
  hipLaunchKernelGGL(dequant_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                     quant, kc, vc, ko, vo, batch, heads, head_dim, S,
                     (int64_t)row_bytes(quant, head_dim));
  PKV_HIP(hipGetLastError());
  return PKV_OK;
}

}  // namespace pkv
