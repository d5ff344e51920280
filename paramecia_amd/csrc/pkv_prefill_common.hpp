// Shared parts of the MFMA prefill-chunk kernels (Q4K, Q8_0, F16 and BF16 caches, the
// Qwen3-Next full-attention shape: 16 query heads, 2 KV heads, head_dim 256): the kernel
// arguments, the work plan (16 query positions x one KV head x one key split per workgroup,
// up to 128 splits by estimated time) and the kernels that merge the key splits' (m, l, o)
// partials. Include-only; every symbol has internal linkage.
//
// Partial layout: part[batch * nsplit + split][kv head][pos * 8 + head of the group][256] in
// tile order (entry i holds element tile_e(i / 16, i % 16)), and ml[same rows]: the row's
// running max m (log2 units) and sum l.
#pragma once
#include "pkv_decode_split.hpp"

namespace pkv {
namespace {

constexpr int kPfWaves = 8;
constexpr int kPfThreads = 64 * kPfWaves;
constexpr int kPosPerWG = 16;  // query positions per workgroup, two per wave
constexpr int kRaw = 3;        // raw block stages in flight
constexpr int kPfTargetWGs = 256;
constexpr float kPfLazy = 8.0f;
constexpr int kNarrowSplits = 16;    // splits the narrow merge takes (all loads in flight)
constexpr int kMaxMergeSplits = 128;  // splits the wide merge takes
constexpr size_t kPfMaxPartBytes = (size_t)256 << 20;

struct PrefillArgs {
  const float *q;  // [B][l][16][256]
  const uint8_t *k, *v;
  int64_t rs_b, rs_t, rs_h;
  int64_t seq_k;     // keys in the cache
  int64_t q_offset;  // query i sees key j iff !causal || j <= i + q_offset
  int l, causal;
  int ntiles, nsplit;  // position tiles; key splits of a tile, each its even share of the
                       // blocks the tile sees (shares of the whole range left the last
                       // splits of a prompt's first tiles empty: 2048 tokens 180 us at 2
                       // splits, 118 us with even ones)
  int ngroups;              // (batch, split, KV head) groups: 2 * nsplit * batch
  float sl2;                // scale * log2(e)
  float *part;  // [B * nsplit][2][l * 8][256] partials in tile order (nsplit > 1)
  float2 *ml;   // [B * nsplit][2][l * 8] their (m, l)
  float *out;   // [B][l][16][256] (nsplit == 1)
};

// A workgroup's tile, KV head, key split and batch row in the 1-D grid of ntiles *
// ngroups workgroups: consecutive workgroups take consecutive (batch, split, KV head)
// groups. The dispatcher deals workgroups to the 8 XCDs round-robin, so with 8 groups
// (the 512-token chunk: 2 KV heads x 4 splits) every workgroup that streams one group's
// key range runs on one XCD and the range is fetched into that XCD's L2 once, not by all
// eight. The tiles go out last first: under the causal limit the last tile sees the most
// keys, and the workgroups dispatched last then are the short ones (a 4001-token prompt,
// 502 workgroups of 1 to 126 blocks on 256 CUs: 451 -> 316 us).
struct PfWork {
  int tile, kvg, split, b;
};
__device__ __forceinline__ PfWork prefill_work(const PrefillArgs &a) {
  const int L = blockIdx.x, grp = L % a.ngroups, z = grp >> 1;
  return PfWork{a.ntiles - 1 - L / a.ngroups, grp & 1, z % a.nsplit, z / a.nsplit};
}

// Merge the key splits: out[b][pos][8 kvg + hh][e] = sum_s o_s 2^(m_s - M) / sum_s l_s 2^(m_s - M).
// One workgroup of 256 threads per 8 rows and batch: 32 threads per row, each taking 8
// consecutive tile-order entries; every split's (m, l) and entries are loaded before any
// is used (nsplit <= kNarrowSplits).
__global__ __launch_bounds__(256) void prefill_merge_kernel(const float *part, const float2 *pml,
                                                            int nsplit, int l, float *out) {
  const int r8 = threadIdx.x >> 5, j = threadIdx.x & 31;
  const int row = blockIdx.x * 8 + r8, b = blockIdx.y;  // row = kvg * l * 8 + pos * 8 + hh
  if (row >= 2 * l * 8) return;
  const int kvg = row / (l * 8), rr = row % (l * 8), pos = rr >> 3, hh = rr & 7;
  const int64_t split_rows = (int64_t)2 * l * 8, row0 = (int64_t)b * nsplit * split_rows + row;
  float2 ml[kNarrowSplits];
  float4 v[kNarrowSplits][2];
#pragma unroll
  for (int s = 0; s < kNarrowSplits; ++s) {
    if (s < nsplit) {
      const int64_t r = row0 + s * split_rows;
      ml[s] = pml[r];
#pragma unroll
      for (int k = 0; k < 2; ++k) v[s][k] = *reinterpret_cast<const float4 *>(part + r * 256 + 8 * j + 4 * k);
    }
  }
  float M = -INFINITY;
#pragma unroll
  for (int s = 0; s < kNarrowSplits; ++s)
    if (s < nsplit) M = fmaxf(M, ml[s].x);
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, L = 0.0f;
#pragma unroll
  for (int s = 0; s < kNarrowSplits; ++s) {
    if (s < nsplit) {
      const float f = (ml[s].x == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(ml[s].x - M);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        acc[4 * k] += f * v[s][k].x;
        acc[4 * k + 1] += f * v[s][k].y;
        acc[4 * k + 2] += f * v[s][k].z;
        acc[4 * k + 3] += f * v[s][k].w;
      }
      L += f * ml[s].y;
    }
  }
  float *orow = out + (((int64_t)b * l + pos) * 16 + 8 * kvg + hh) * 256;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int idx = 8 * j + k;
    orow[tile_e(idx >> 4, idx & 15)] = L > 0.0f ? acc[k] / L : 0.0f;
  }
}

// The same for up to kMaxMergeSplits splits (a short chunk over many keys): one workgroup
// of 8 groups of 32 threads per row and batch. Group sg takes splits sg, sg + 8, ...: up
// to kPer of them, every load issued before any is used; the groups' sums meet in LDS.
// (2 x 33 tokens over 3033 keys at 20 splits: 41.3 us with 16 loads a group, 35.4 with 4.)
template <int kPer>
__global__ __launch_bounds__(256) void prefill_merge_wide_kernel(const float *part,
                                                                 const float2 *pml, int nsplit,
                                                                 int l, float *out) {
  __shared__ __attribute__((aligned(16))) float acc_s[8][256];
  __shared__ float2 ml_s[8];
  const int sg = threadIdx.x >> 5, j = threadIdx.x & 31;
  const int row = blockIdx.x, b = blockIdx.y;
  const int kvg = row / (l * 8), rr = row % (l * 8), pos = rr >> 3, hh = rr & 7;
  const int64_t split_rows = (int64_t)2 * l * 8, row0 = (int64_t)b * nsplit * split_rows + row;
  float2 ml[kPer];
  float4 v[kPer][2];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int s = sg + 8 * i;
    const bool ok = s < nsplit;  // past the splits: split 0's row, with no weight
    const int64_t r = row0 + (ok ? s : 0) * split_rows;
    const float2 t = pml[r];
    ml[i] = ok ? t : float2{-INFINITY, 0.0f};
#pragma unroll
    for (int k = 0; k < 2; ++k) v[i][k] = *reinterpret_cast<const float4 *>(part + r * 256 + 8 * j + 4 * k);
  }
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < kPer; ++i) m = fmaxf(m, ml[i].x);
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, L = 0.0f;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    if (ml[i].x == -INFINITY) continue;
    const float f = __builtin_amdgcn_exp2f(ml[i].x - m);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      acc[4 * k] += f * v[i][k].x;
      acc[4 * k + 1] += f * v[i][k].y;
      acc[4 * k + 2] += f * v[i][k].z;
      acc[4 * k + 3] += f * v[i][k].w;
    }
    L += f * ml[i].y;
  }
  *reinterpret_cast<float4 *>(&acc_s[sg][8 * j]) = float4{acc[0], acc[1], acc[2], acc[3]};
  *reinterpret_cast<float4 *>(&acc_s[sg][8 * j + 4]) = float4{acc[4], acc[5], acc[6], acc[7]};
  if (j == 0) ml_s[sg] = float2{m, L};
  __syncthreads();
  float M = -INFINITY, Lt = 0.0f, o = 0.0f;
#pragma unroll
  for (int g = 0; g < 8; ++g) M = fmaxf(M, ml_s[g].x);
  const int idx = threadIdx.x;
#pragma unroll
  for (int g = 0; g < 8; ++g) {
    const float f = (ml_s[g].x == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(ml_s[g].x - M);
    o += f * acc_s[g][idx];
    Lt += f * ml_s[g].y;
  }
  out[(((int64_t)b * l + pos) * 16 + 8 * kvg + hh) * 256 + tile_e(idx >> 4, idx & 15)] =
      Lt > 0.0f ? o / Lt : 0.0f;
}

}  // namespace

// Bytes of an nsplit-way plan's partials.
static inline size_t prefill_part_bytes(int batch, int nsplit, int l) {
  return (size_t)batch * nsplit * 2 * l * 8 * 258 * sizeof(float);
}

// The number of key splits: the one with the least estimated time, in units of a block
// (32 keys) of one workgroup, of which 256 run at a time (one per CU). A workgroup takes its
// blocks + kPfFixed. Up to 256 workgroups end with the longest one. Of more, dispatched
// longest first, the last round's each follow one of the round before, the two as long as
// those at the rounds' boundary. The merge writes and reads its partials. Only splits that
// leave no share of the last tile empty are looked at.
// Measured with every split over 2 to 4096 tokens, 0 to 60000 cached, 1 and 2 rows of Q4K, Q8_0
// and F16 (696 shapes): the split taken is 0.4% slower than the best one in the mean, over 10%
// in 3 shapes. Whole rounds of mean workgroups and merges twice as dear had 1.3% and 32 (Q8_0
// 700 tokens after 500 64.1 us at 3 splits, 72.3 at the 2 taken then). A few tokens over a
// long cache take as many splits as give every CU a workgroup: 5 tokens over 20016 keys 98.8 us
// at 16 splits, 24.5 at 126. The partials take kPfMaxPartBytes at most: beyond lie chunks of
// many rows that fill the GPU without a split.
static inline int prefill_splits(const AttnArgs &a, int ntiles, int nblk) {
  constexpr double kPfFixed = 3.5;  // q, the first block's latency, the epilogue
  // the merge's launch, and bytes of partials in a block's time: fewer where one round of
  // workgroups writes them at its end, half past kMergeNear
  constexpr double kMergeFixed = 0.9, kMergeBytes1 = 5e6, kMergeBytes = 8e6, kMergeNear = 64e6;
  // blocks of the first and the last tile (the causal limit cuts the first ones')
  int nb0 = nblk, nb1 = nblk;
  if (a.causal) {
    auto seen = [&](int64_t keys) { return (int)(((keys < a.seq_k ? keys : a.seq_k) + 31) / 32); };
    nb0 = seen(a.q_offset + (a.l < kPosPerWG ? a.l : kPosPerWG));
    nb1 = seen(a.q_offset + a.l);
  }
  int best = 1;
  double best_t = 1e30;
  for (int ns = 1; ns <= kMaxMergeSplits && ns <= (nb1 > 0 ? nb1 : 1); ++ns) {
    const size_t bytes = ns > 1 ? prefill_part_bytes(a.batch, ns, a.l) : 0;
    if (bytes > kPfMaxPartBytes) break;
    const int share = (nb1 + ns - 1) / ns;
    if (ns > 1 && (nb1 + share - 1) / share != ns) continue;
    const double longest = share + kPfFixed, shortest = (nb0 + ns - 1) / ns + kPfFixed;
    const double wgs = 2.0 * ntiles * a.batch * ns;
    double t = longest;
    if (wgs > kPfTargetWGs) {
      const double full = (double)(int64_t)((wgs - 1) / kPfTargetWGs);  // rounds before the last
      auto length = [&](double rounds) { return longest - (longest - shortest) * rounds * kPfTargetWGs / wgs; };
      const double sum = (full - 1) * 0.5 * (longest + length(full - 1)) + 2 * length(full);
      t = sum > t ? sum : t;
    }
    if (ns > 1)
      t += kMergeFixed + bytes / (wgs <= kPfTargetWGs ? kMergeBytes1 : kMergeBytes) +
           (bytes > kMergeNear ? (bytes - kMergeNear) / kMergeBytes : 0.0);
    if (t < best_t) {
      best_t = t;
      best = ns;
    }
  }
  return best;
}

// Scratch by which a no-alloc call is accepted: the partials of 256 workgroups' worth of splits
// (16 at most).
static inline size_t prefill_accept_bytes(const AttnArgs &a, int ntiles, int nblk) {
  const int base = ntiles * 2 * a.batch;
  int need = (kPfTargetWGs + base - 1) / base;
  need = need > 16 ? 16 : need;
  need = need > nblk ? (nblk > 0 ? nblk : 1) : need;
  return need > 1 ? prefill_part_bytes(a.batch, need, a.l) : 0;
}

// The split merge after a prefill kernel that wrote partials (nsplit > 1).
static inline int prefill_merge(const PrefillArgs &d, int batch, hipStream_t s) {
  if (d.nsplit <= 1) return PKV_OK;
  if (d.nsplit <= kNarrowSplits)
    hipLaunchKernelGGL(prefill_merge_kernel, dim3((unsigned)((2 * d.l * 8 + 7) / 8), (unsigned)batch),
                       dim3(256), 0, s, d.part, d.ml, d.nsplit, d.l, d.out);
  else {
    const auto wide = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3((unsigned)(2 * d.l * 8), (unsigned)batch), dim3(256), 0, s, d.part,
                         d.ml, d.nsplit, d.l, d.out);
    };
    if (d.nsplit <= 32) wide(prefill_merge_wide_kernel<4>);
    else if (d.nsplit <= 64) wide(prefill_merge_wide_kernel<8>);
    else wide(prefill_merge_wide_kernel<kMaxMergeSplits / 8>);
  }
  PKV_HIP(hipGetLastError());
  return PKV_OK;
}

// Plan and run a prefill chunk over 32-key blocks: launch(d, grid) enqueues the attention
// kernel, the merge follows. accept_bytes: scratch that a no-alloc call of this shape has to have
// besides.
// A no-alloc call uses the splits of an allocating one, so that the two give the same bits.
// Where their partials exceed its memory, position tiles go through it a group at a time, each a
// chunk of its own over the same keys. (Fewer splits that fit took 64 us for 32 tokens over
// 20000 Q4K keys, in place of 46.6.)
template <typename Launch>
static inline int prefill_run(const AttnArgs &a, float sl2, Workspace &ws, hipStream_t s,
                              size_t accept_bytes, Launch launch) {
  const int ntiles = (a.l + kPosPerWG - 1) / kPosPerWG, nblk = (int)((a.seq_k + 31) / 32);
  if (ws.fixed) {
    const size_t bytes = prefill_accept_bytes(a, ntiles, nblk);
    if (const int rc = ws.reserve(bytes > accept_bytes ? bytes : accept_bytes)) return rc;
  }
  const int nsplit = prefill_splits(a, ntiles, nblk);
  auto run = [&](const AttnArgs &c) -> int {
    PrefillArgs d;
    d.q = c.q;
    d.k = c.k;
    d.v = c.v;
    d.rs_b = c.rs.b;
    d.rs_t = c.rs.t;
    d.rs_h = c.rs.h;
    d.seq_k = c.seq_k;
    d.q_offset = c.q_offset;
    d.l = c.l;
    d.causal = c.causal ? 1 : 0;
    d.sl2 = sl2;
    d.ntiles = (c.l + kPosPerWG - 1) / kPosPerWG;
    d.nsplit = nsplit;
    d.ngroups = 2 * nsplit * c.batch;
    d.out = c.out;
    d.part = nullptr;
    d.ml = nullptr;
    if (nsplit > 1) {
      d.part = static_cast<float *>(ws.ptr);
      d.ml = reinterpret_cast<float2 *>(d.part + (size_t)c.batch * nsplit * 2 * c.l * 8 * 256);
    }
    launch(d, dim3((unsigned)(d.ntiles * d.ngroups)));
    PKV_HIP(hipGetLastError());
    return prefill_merge(d, c.batch, s);
  };
  const size_t part_bytes = nsplit > 1 ? prefill_part_bytes(a.batch, nsplit, a.l) : 0;
  if (!ws.fixed) {
    if (const int rc = ws.reserve(part_bytes)) return rc;
    return run(a);
  }
  if (part_bytes <= kNoallocBytes) return run(a);
  static_assert((size_t)kMaxMergeSplits * 2 * kPosPerWG * 8 * 258 * sizeof(float) <= kNoallocBytes,
                "a tile's partials fit");
  const int step = (int)(kNoallocBytes / prefill_part_bytes(1, nsplit, kPosPerWG)) * kPosPerWG;
  const int64_t q_row = (int64_t)a.num_heads * a.head_dim;
  for (int b = 0; b < a.batch; ++b)
    for (int p0 = 0; p0 < a.l; p0 += step) {
      AttnArgs c = a;
      c.batch = 1;
      c.l = a.l - p0 < step ? a.l - p0 : step;
      c.k = a.k + b * a.rs.b;
      c.v = a.v + b * a.rs.b;
      c.q = a.q + ((int64_t)b * a.l + p0) * q_row;
      c.out = a.out + ((int64_t)b * a.l + p0) * q_row;
      c.q_offset = a.q_offset + p0;
      if (const int rc = run(c)) return rc;
    }
  return PKV_OK;
}

}  // namespace pkv
