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
// of V. kWide: 16-byte loads from both tensors.
template <int kL, bool kWide>
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
  if (kWide && e0 + E <= a.head_dim) {
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

  q4k_quantize_group<kL>(x, r, [&] { return row_ptr(a, p, t, b, h) + (int64_t)sb * 144; }, active);
}

// Four elements of a row per lane: 16-byte loads where kWide (head_dim a multiple of 4, K
// and V 16-byte aligned), else one by one. U counts quads: 32 bits but for appends of 2^31
// quads and more. Quad i's tensor p, row (t, b, h) and elements e .. e + 3; false past the end.
struct Quad {
  float x[4];
  int p, b, h, e;
  int64_t t;
};
template <bool kWide, typename U>
__device__ __forceinline__ bool load_quad(const AppendArgs &a, U quads_per_tensor, U i, Quad &q) {
  if (i >= 2 * quads_per_tensor) return false;
  q.p = i >= quads_per_tensor;
  const U u = q.p ? i - quads_per_tensor : i;
  const U per_row = (U)a.padded >> 2, r = u / per_row;
  q.e = (int)(u - r * per_row) * 4;
  const U rh = r / (U)a.heads, t = rh / (U)a.batch;
  q.h = (int)(r - rh * (U)a.heads);
  q.t = (int64_t)t;
  q.b = (int)(rh - t * (U)a.batch);
  const float *src = a.src[q.p];
  if constexpr (kWide) {
    float4 f = {0.f, 0.f, 0.f, 0.f};
    if (q.e < a.head_dim)
      f = *reinterpret_cast<const float4 *>(
          src + (((int64_t)q.b * a.heads + q.h) * a.n + q.t) * a.head_dim + q.e);
    q.x[0] = f.x;
    q.x[1] = f.y;
    q.x[2] = f.z;
    q.x[3] = f.w;
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) q.x[k] = load_elem(src, a, q.t, q.b, q.h, q.e + k);
  }
  return true;
}

// Q8_0 (BlockQ8_0::from_float): 8 lanes per 32-element block, four elements each, so that a
// wave reads 1 KB and writes 272 bytes in a row. The block's largest |x| is exact in any
// order (NaN dropped, as f32::max does). One lane per block, with 32 scalar loads and 17
// 2-byte stores, took 11.0 us for 512 tokens of the model's shape (2.7 MB), this form 3.3 us.
// With 64-bit counts the lanes go on by the grid's size: a launch holds fewer than 2^32.
template <bool kWide, typename U>
__device__ __forceinline__ bool q8_0_append_quad(const AppendArgs &a, U quads_per_tensor, U i) {
  Quad q;
  if (!load_quad<kWide, U>(a, quads_per_tensor, i, q)) return false;
  int32_t key = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int32_t v = (q.x[k] != q.x[k]) ? 0 : (int32_t)(f2u(q.x[k]) & 0x7FFFFFFFu);
    key = v > key ? v : key;
  }
#pragma unroll
  for (int o = 1; o < 8; o <<= 1) {
    const int32_t v = __shfl_xor(key, o, 8);
    key = v > key ? v : key;
  }
  const float d = u2f((uint32_t)key) / 127.0f;
  const float id = (d != 0.0f) ? 1.0f / d : 0.0f;
  uint32_t w = 0u;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    w |= (uint32_t)(uint8_t)rs_as_i8(__builtin_roundf(q.x[k] * id)) << (8 * k);
  uint8_t *blk = row_ptr(a, q.p, q.t, q.b, q.h) + (q.e >> 5) * 34;
  uint16_t *o = reinterpret_cast<uint16_t *>(blk + 2 + (q.e & 31));
  o[0] = (uint16_t)w;
  o[1] = (uint16_t)(w >> 16);
  if ((q.e & 31) == 0) *reinterpret_cast<uint16_t *>(blk) = f32_to_f16(d);
  return true;
}
template <bool kWide, typename U>
__global__ __launch_bounds__(256) void q8_0_append_kernel(AppendArgs a, U quads_per_tensor) {
  U i = (U)blockIdx.x * 256 + threadIdx.x;
  if constexpr (sizeof(U) == 4) {
    q8_0_append_quad<kWide, U>(a, quads_per_tensor, i);
  } else {
    while (q8_0_append_quad<kWide, U>(a, quads_per_tensor, i)) i += (U)gridDim.x * 256;
  }
}

// F16 / BF16 rows: round-to-nearest-even conversion, four elements a lane (4096 tokens of
// the model's shape 20.9 us one by one, 9.5 now). Rows of a head_dim that is no multiple
// of 4 go element by element.
template <bool BF, bool kWide>
__global__ __launch_bounds__(256) void half_append_quads_kernel(AppendArgs a,
                                                                uint32_t quads_per_tensor) {
  Quad q;
  if (!load_quad<kWide, uint32_t>(a, quads_per_tensor, blockIdx.x * 256 + threadIdx.x, q)) return;
  uint32_t y[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) y[k] = BF ? f32_to_bf16(q.x[k]) : f32_to_f16(q.x[k]);
  *reinterpret_cast<uint2 *>(row_ptr(a, q.p, q.t, q.b, q.h) + 2 * q.e) =
      uint2{y[0] | (y[1] << 16), y[2] | (y[3] << 16)};
}
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
  // 16-byte loads: rows of a multiple of 4 elements from aligned tensors
  const bool wide = (a.head_dim & 3) == 0 && ((reinterpret_cast<uintptr_t>(a.src[0]) |
                                               reinterpret_cast<uintptr_t>(a.src[1])) & 15) == 0;
  if (quant == PKV_QUANT_Q4K) {
    // 8 kL lanes per superblock: split each sub-block's fit over more lanes while the
    // append has too few superblocks to give every SIMD a wave (a workgroup of 256 lanes
    // per superblock, the fused decode's quantizer, took 6.8 us for 1 to 64 tokens of the
    // model's shape and 11.1 for 256 where 4 lanes per sub-block take 6.0 and 6.2)
    const int nsb = a.padded / 256;
    const int64_t units = rows * nsb;
    const int kl = 2 * units <= kQ4kAppendLanes4Max ? 4 : (2 * units <= kQ4kAppendLanes2Max ? 2 : 1);
    const int64_t threads = 2 * units * 8 * kl;
    const dim3 grid((unsigned)((threads + 255) / 256));
    const auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, a, units, nsb); };
    if (kl == 4) go(wide ? q4k_append_kernel<4, true> : q4k_append_kernel<4, false>);
    else if (kl == 2) go(wide ? q4k_append_kernel<2, true> : q4k_append_kernel<2, false>);
    else go(wide ? q4k_append_kernel<1, true> : q4k_append_kernel<1, false>);
  } else {
    const bool q8 = quant == PKV_QUANT_Q8_0, bf = quant == PKV_QUANT_BF16;
    const int64_t elems = rows * a.padded, blocks = (2 * (elems / 4) + 255) / 256;
    const bool fit32 = elems / 2 < (1ll << 31);
    const uint32_t quads = (uint32_t)(elems / 4);
    const dim3 grid((unsigned)blocks), t(256);
    // 8-byte stores: rows at multiples of 4 elements
    const bool half_quads = (a.padded & 3) == 0 && fit32;
    if (q8 && !fit32)
      hipLaunchKernelGGL((q8_0_append_kernel<false, uint64_t>), dim3(1u << 20), t, 0, s, a, (uint64_t)elems / 4);
    else if (q8 && wide)
      hipLaunchKernelGGL((q8_0_append_kernel<true, uint32_t>), grid, t, 0, s, a, quads);
    else if (q8)
      hipLaunchKernelGGL((q8_0_append_kernel<false, uint32_t>), grid, t, 0, s, a, quads);
    else if (half_quads && bf && wide)
      hipLaunchKernelGGL((half_append_quads_kernel<true, true>), grid, t, 0, s, a, quads);
    else if (half_quads && bf)
      hipLaunchKernelGGL((half_append_quads_kernel<true, false>), grid, t, 0, s, a, quads);
    else if (half_quads && wide)
      hipLaunchKernelGGL((half_append_quads_kernel<false, true>), grid, t, 0, s, a, quads);
    else if (half_quads)
      hipLaunchKernelGGL((half_append_quads_kernel<false, false>), grid, t, 0, s, a, quads);
    else if (bf)
      hipLaunchKernelGGL(half_append_kernel<true>, dim3((unsigned)((2 * elems + 255) / 256)), t, 0,
                         s, a, elems);
    else
      hipLaunchKernelGGL(half_append_kernel<false>, dim3((unsigned)((2 * elems + 255) / 256)), t, 0,
                         s, a, elems);
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
