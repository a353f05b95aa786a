// Backward of the trilinear embedding gather: the gradient of the corner
// embedding table from the gradient of the gathered embeddings.
//
// Forward (encoder.py:582-590, geometry.py:195-200): out[m] = sum_c w_c(m) *
// values[feats[v_m][c]].  Its adjoint, which torch forms for the reference as
// the backward of F.embedding (an index-add into values.weight), is
//   grad_values[k] = sum over (v, c) with feats[v][c] == k of
//                    sum over samples m in voxel v of w_c(m) * grad_out[m].
// The reference's index-add uses atomics, so its summation order (and last
// bits) vary run to run.  Here the sums are deterministic and atomic-free:
//
//   1. sort the samples by voxel (stable radix sort; slot order within a
//      voxel) and find each voxel's segment by binary search;
//   2. one wavefront per voxel: lane (c, j) accumulates w_c(m) * grad_out[m]
//      over the voxel's samples for corner c and features 4j.. (+32 ...),
//      in sample order, into G[v][c] -- the per-(voxel, corner) partials;
//   3. sort the (voxel, corner) incidences by corner key the same way, and
//      sum each key's <= 8 partials G[v][c] in incidence order.  The
//      incidence order depends only on the scene's corner keys, so a caller
//      that differentiates the same scene repeatedly computes it once (a
//      "plan": the sorted incidences and the key segments) and passes it.
//
// The corner weights are the forward gather's, computed with the same
// operations, so the backward is the exact adjoint of the forward's weights.
// Traffic: the sample gradients are read once (plus 12 bytes of position
// and 8 of sort keys per sample); G is N * 8 * D floats written once and
// read once; the table gradient is written once.
#include <algorithm>

#include "common.h"

namespace nsvf {
namespace {

constexpr int kBlock = 256;

inline int64_t align256(int64_t b) { return (b + 255) & ~int64_t(255); }

// bits needed for keys in [0, n]
inline int key_bits(int64_t n) {
  int b = 1;
  while (b < 31 && (int64_t(1) << b) <= n) ++b;
  return b;
}

// Stable radix sort of (key, index) pairs, 8 bits per pass: the digits of each
// tile of kTile items are counted, every digit's counts summed over the tiles,
// and the items written behind those of smaller digits and earlier tiles.  The
// keys are those of a caller's array (anything outside [0, limit) is `limit`)
// and the values 0, 1, ..., so the first pass reads that array itself.  For
// 800,003 samples of 100k voxels (17 bits, three passes) 64 us; a
// merge sort of the pairs took 163.
constexpr int kItems = 8;                // per thread
constexpr int kTile = kBlock * kItems;

// A tile's keys, wave by wave in item order: item k of lane l of wave w is
// 64 (kItems w + k) + l.
template <bool kFirst>
__device__ __forceinline__ bool sort_key(const void* __restrict__ src, int64_t n, int32_t limit,
                                         int k, uint32_t* key, int64_t* i) {
  *i = int64_t(blockIdx.x) * kTile + 64 * (kItems * (threadIdx.x >> 6) + k) + (threadIdx.x & 63);
  *key = 0;
  if (*i >= n) return false;
  if constexpr (kFirst) {
    const int32_t v = static_cast<const int32_t*>(src)[*i];
    *key = uint32_t(v < 0 || v >= limit ? limit : v);
  } else {
    *key = static_cast<const uint32_t*>(src)[*i];
  }
  return true;
}

// counts[digit][tile]
template <bool kFirst>
__global__ __launch_bounds__(kBlock) void digit_count_kernel(const void* __restrict__ src,
                                                             int64_t n, int32_t limit, int shift,
                                                             uint32_t* __restrict__ counts) {
  __shared__ uint32_t bin[256];
  bin[threadIdx.x] = 0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    uint32_t key;
    int64_t i;
    if (sort_key<kFirst>(src, n, limit, k, &key, &i)) atomicAdd(&bin[key >> shift & 255], 1u);
  }
  __syncthreads();
  counts[int64_t(threadIdx.x) * gridDim.x + blockIdx.x] = bin[threadIdx.x];
}

// Exclusive sums over the 256 threads of a block; *all: their total.
__device__ __forceinline__ uint32_t block_exclusive(uint32_t v, uint32_t* wave_sums,
                                                    uint32_t* all) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t sum = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t left = __shfl_up(sum, d, 64);
    if (lane >= d) sum += left;
  }
  if (lane == 63) wave_sums[wave] = sum;
  __syncthreads();
  uint32_t before = 0;
  *all = 0;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) {
    before += w < wave ? wave_sums[w] : 0;
    *all += wave_sums[w];
  }
  __syncthreads();
  return before + sum - v;
}

// Block d: counts[d][*] to exclusive sums, totals[d] their sum.
__global__ __launch_bounds__(kBlock) void digit_scan_kernel(uint32_t* __restrict__ counts,
                                                            int64_t tiles,
                                                            uint32_t* __restrict__ totals) {
  __shared__ uint32_t wave_sums[kBlock / 64];
  uint32_t* row = counts + int64_t(blockIdx.x) * tiles;
  uint32_t carry = 0;
  for (int64_t t0 = 0; t0 < tiles; t0 += kBlock) {
    const int64_t t = t0 + threadIdx.x;
    uint32_t all;
    const uint32_t sum = block_exclusive(t < tiles ? row[t] : 0, wave_sums, &all);
    if (t < tiles) row[t] = carry + sum;
    carry += all;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

template <bool kFirst>
__global__ __launch_bounds__(kBlock) void digit_scatter_kernel(
    const void* __restrict__ src, const int32_t* __restrict__ vals, int64_t n, int32_t limit,
    int shift, const uint32_t* __restrict__ counts, const uint32_t* __restrict__ totals,
    uint32_t* __restrict__ keys_out, int32_t* __restrict__ vals_out) {
  __shared__ uint32_t at[kBlock / 64][256], wave_sums[kBlock / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) at[w][threadIdx.x] = 0;
  __syncthreads();
  uint32_t key[kItems], rank[kItems];
  int32_t val[kItems];
  bool have[kItems];
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    int64_t i;
    have[k] = sort_key<kFirst>(src, n, limit, k, &key[k], &i);
    val[k] = kFirst ? int32_t(i) : have[k] ? vals[i] : 0;
  }
  // an item's rank among the wave's items of its digit
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    const uint32_t d = key[k] >> shift & 255;
    uint64_t same = __ballot(have[k]);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint64_t ones = __ballot(d >> b & 1);
      same &= d >> b & 1 ? ones : ~ones;
    }
    const uint32_t lower = uint32_t(__popcll(same & ((uint64_t(1) << lane) - 1)));
    rank[k] = at[wave][d] + lower;
    wave_sync();
    if (have[k] && lower == 0) at[wave][d] += uint32_t(__popcll(same));
    wave_sync();
  }
  __syncthreads();
  // digit threadIdx.x: the first place of each wave's items
  uint32_t all;
  uint32_t first = block_exclusive(totals[threadIdx.x], wave_sums, &all) +
                   counts[int64_t(threadIdx.x) * gridDim.x + blockIdx.x];
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) {
    const uint32_t c = at[w][threadIdx.x];
    at[w][threadIdx.x] = first;
    first += c;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kItems; ++k)
    if (have[k]) {
      const uint32_t pos = at[wave][key[k] >> shift & 255] + rank[k];
      keys_out[pos] = key[k];
      vals_out[pos] = val[k];
    }
}

inline int64_t sort_tiles(int64_t n) { return ceil_div(n, kTile); }
inline int64_t sort_counts(int64_t n) { return 256 * sort_tiles(n) + 256; }

// Sorts items 0 .. n - 1 by src[i] (0 <= key <= limit) into keys, vals; the
// other pair and counts [sort_counts(n)] are scratch.
void sort_by_key(const int32_t* src, int64_t n, int32_t limit, uint32_t* keys, int32_t* vals,
                 uint32_t* keys2, int32_t* vals2, uint32_t* counts, hipStream_t st) {
  if (n == 0) return;
  const int passes = int(ceil_div(key_bits(limit), 8));
  const dim3 grid{unsigned(sort_tiles(n))}, block{kBlock};
  uint32_t* totals = counts + 256 * sort_tiles(n);
  const void* in = src;
  const int32_t* in_vals = nullptr;
  for (int p = 0; p < passes; ++p) {
    const bool to_out = (passes - 1 - p) % 2 == 0;   // the last pass ends in keys, vals
    uint32_t* k = to_out ? keys : keys2;
    int32_t* v = to_out ? vals : vals2;
    hipLaunchKernelGGL(p == 0 ? digit_count_kernel<true> : digit_count_kernel<false>, grid, block,
                       0, st, in, n, limit, 8 * p, counts);
    hipLaunchKernelGGL(digit_scan_kernel, dim3(256), block, 0, st, counts, sort_tiles(n), totals);
    hipLaunchKernelGGL(p == 0 ? digit_scatter_kernel<true> : digit_scatter_kernel<false>, grid,
                       block, 0, st, in, in_vals, n, limit, 8 * p, counts, totals, k, v);
    in = k;
    in_vals = v;
  }
}

struct GradWorkspace {
  uint32_t* keys;      // [M] voxel of each sample (N for unused), sorted
  uint32_t* keys2;
  int32_t* vals;       // [M] sample ids
  int32_t* vals2;
  int32_t* seg;        // [N + 1] voxel segment starts in the sorted samples
  uint32_t* ikeys;     // [8N] corner key of each (voxel, corner), sorted
  uint32_t* ikeys2;
  int32_t* ivals;      // [8N] incidence ids v * 8 + c
  int32_t* ivals2;
  int32_t* kseg;       // [K + 1] key segment starts in the sorted incidences
  float* partial;      // [8N, D] per-(voxel, corner) partial gradients
  uint32_t* counts;    // the sorts' digit counts
  int64_t total;
};

void layout(int64_t M, int64_t N, int64_t K, int D, char* base, GradWorkspace* w) {
  int64_t o = 0;
  auto take = [&](int64_t bytes) {
    char* p = base ? base + o : nullptr;
    o += align256(bytes);
    return p;
  };
  w->keys = reinterpret_cast<uint32_t*>(take(M * 4));
  w->keys2 = reinterpret_cast<uint32_t*>(take(M * 4));
  w->vals = reinterpret_cast<int32_t*>(take(M * 4));
  w->vals2 = reinterpret_cast<int32_t*>(take(M * 4));
  w->seg = reinterpret_cast<int32_t*>(take((N + 1) * 4));
  w->ikeys = reinterpret_cast<uint32_t*>(take(8 * N * 4));
  w->ikeys2 = reinterpret_cast<uint32_t*>(take(8 * N * 4));
  w->ivals = reinterpret_cast<int32_t*>(take(8 * N * 4));
  w->ivals2 = reinterpret_cast<int32_t*>(take(8 * N * 4));
  w->kseg = reinterpret_cast<int32_t*>(take((K + 1) * 4));
  w->partial = reinterpret_cast<float*>(take(8 * N * int64_t(D) * 4));
  w->counts = reinterpret_cast<uint32_t*>(take(sort_counts(std::max(M, 8 * N)) * 4));
  w->total = o;
}

// seg[v] = first position of a key >= v in sorted[0, n), v = 0..nseg-1.
__global__ __launch_bounds__(kBlock) void segment_starts_kernel(
    const uint32_t* __restrict__ sorted, int64_t n, int64_t nseg, int32_t* __restrict__ seg) {
  const int64_t v = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (v >= nseg) return;
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (int64_t(sorted[mid]) < v)
      lo = mid + 1;
    else
      hi = mid;
  }
  seg[v] = int32_t(lo);
}

// One wavefront per voxel; lane = 8 * corner + j.  Feature float4 groups
// q = j, j + 8, ... < D / 4 (Q = 1, 2 or 4 of them cover D <= 32, 64, 128).
// Bound: the latency of a voxel's chain sample id -> gradient row.  Eight
// samples go together: lane j of each corner's group forms the weight of the
// eighth it owns, and the eight gradient rows are in flight at once; the sums
// stay in sample order.  100k voxels of 8 samples, D = 32: 201 -> 78 us.
template <int Q>
__global__ __launch_bounds__(kBlock) void voxel_corner_kernel(
    const int32_t* __restrict__ seg, const int32_t* __restrict__ order,
    const float* __restrict__ xyz, const float* __restrict__ centers, float voxel_size,
    const float* __restrict__ grad_out, int D, int64_t N, float* __restrict__ partial) {
  constexpr int R = Q == 4 ? 4 : 8;   // rows in flight
  const int64_t v =
      int64_t(blockIdx.x) * (kBlock / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (v >= N) return;
  const int lane = threadIdx.x & 63;
  const int c = lane >> 3, j = lane & 7;
  const int DQ = D >> 2;
  const float cx = centers[v * 3 + 0], cy = centers[v * 3 + 1], cz = centers[v * 3 + 2];
  float4 acc[Q];
#pragma unroll
  for (int t = 0; t < Q; ++t) acc[t] = make_float4(0.f, 0.f, 0.f, 0.f);
  const int32_t s0 = seg[v], s1 = seg[v + 1];
  for (int32_t i0 = s0; i0 < s1; i0 += 64) {
    const int n = min(s1 - i0, 64);
    const int32_t mine = order[i0 + min(lane, n - 1)];
    for (int b = 0; b < n; b += 8) {
      // corner weight of the forward gather: p = (x - c) / vs + 0.5,
      // w = (wx * wy) * wz
      const int64_t mj = __shfl(mine, min(b + j, n - 1), 64);
      const float px = (xyz[mj * 3 + 0] - cx) / voxel_size + 0.5f;
      const float py = (xyz[mj * 3 + 1] - cy) / voxel_size + 0.5f;
      const float pz = (xyz[mj * 3 + 2] - cz) / voxel_size + 0.5f;
      const float wx = (c & 4) ? px : 1.0f - px;
      const float wy = (c & 2) ? py : 1.0f - py;
      const float wz = (c & 1) ? pz : 1.0f - pz;
      const float wj = (wx * wy) * wz;
      const int nb = min(n - b, 8);
#pragma unroll
      for (int r0 = 0; r0 < 8; r0 += R) {
        float4 x[R][Q];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int64_t m = __builtin_amdgcn_readlane(mine, min(b + r0 + r, n - 1));
          const float4* g = reinterpret_cast<const float4*>(grad_out + m * D);
#pragma unroll
          for (int t = 0; t < Q; ++t)
            if (j + 8 * t < DQ) x[r][t] = g[j + 8 * t];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if (r0 + r >= nb) break;
          const float w = __shfl(wj, (lane & 56) + r0 + r, 64);
#pragma unroll
          for (int t = 0; t < Q; ++t) {
            acc[t].x = acc[t].x + w * x[r][t].x;
            acc[t].y = acc[t].y + w * x[r][t].y;
            acc[t].z = acc[t].z + w * x[r][t].z;
            acc[t].w = acc[t].w + w * x[r][t].w;
          }
        }
      }
    }
  }
  float4* out = reinterpret_cast<float4*>(partial + (v * 8 + c) * D);
#pragma unroll
  for (int t = 0; t < Q; ++t) {
    const int q = j + 8 * t;
    if (q < DQ) out[q] = acc[t];
  }
}

// Thread per (key, float4 group): sum of the key's (voxel, corner) partials
// in incidence order.
__global__ __launch_bounds__(kBlock) void key_sum_kernel(const int32_t* __restrict__ kseg,
                                                         const int32_t* __restrict__ inc,
                                                         const float* __restrict__ partial,
                                                         int64_t K, int D,
                                                         float* __restrict__ grad_values) {
  const int64_t t = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  const int DQ = D >> 2;
  if (t >= K * DQ) return;
  const int64_t k = t / DQ;
  const int q = int(t - k * DQ);
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int32_t i = kseg[k]; i < kseg[k + 1]; ++i) {
    const float4 x = reinterpret_cast<const float4*>(partial + int64_t(inc[i]) * D)[q];
    acc.x = acc.x + x.x;
    acc.y = acc.y + x.y;
    acc.z = acc.z + x.z;
    acc.w = acc.w + x.w;
  }
  reinterpret_cast<float4*>(grad_values + k * D)[q] = acc;
}

// Plan layout: [8N] sorted incidence ids, then [K + 1] key segment starts.
inline int64_t plan_bytes(int64_t N, int64_t K) { return align256(8 * N * 4) + (K + 1) * 4; }

// Step 3's incidence order into plan (ivals: 8N ids, kseg: K + 1 starts),
// using the workspace's incidence buffers and sort space.
int build_plan(const int32_t* feats, int64_t N, int64_t K, const GradWorkspace& w,
               int32_t* ivals, int32_t* kseg, hipStream_t st) {
  sort_by_key(feats, 8 * N, int32_t(K), w.ikeys, ivals, w.ikeys2, w.ivals2, w.counts, st);
  hipLaunchKernelGGL(segment_starts_kernel, dim3(unsigned(ceil_div(K + 1, kBlock))), dim3(kBlock),
                     0, st, w.ikeys, 8 * N, K + 1, kseg);
  return check_launch("gather backward plan");
}

int check_sizes(const char* what, int64_t M, int64_t N, int64_t K, int D) {
  if (M < 0 || N <= 0 || K <= 0 || D <= 0) return set_error(NSVF_EINVAL, "%s: bad size", what);
  if (D % 4 != 0 || D > 128)
    return set_error(NSVF_EINVAL, "%s: D=%d (a multiple of 4, <= 128)", what, D);
  if (M >= (int64_t(1) << 31) || 8 * N >= (int64_t(1) << 31) || K >= (int64_t(1) << 30))
    return set_error(NSVF_EINVAL, "%s: size beyond 32-bit indexing", what);
  return NSVF_OK;
}

}  // namespace
}  // namespace nsvf

using namespace nsvf;

extern "C" {

int64_t nsvf_trilinear_gather_backward_plan_bytes(int64_t N, int64_t K) {
  clear_error();
  if (N <= 0 || K <= 0) {
    set_error(NSVF_EINVAL, "trilinear_gather_backward_plan_bytes: bad size");
    return -1;
  }
  return plan_bytes(N, K);
}

int nsvf_trilinear_gather_backward_plan(const int32_t* feats, int64_t N, int64_t K, void* plan,
                                        int64_t plan_bytes_given, void* workspace,
                                        int64_t workspace_bytes, void* stream) {
  clear_error();
  if (int rc = check_sizes("trilinear_gather_backward_plan", 0, N, K, 4)) return rc;
  if (!feats || !plan || !workspace)
    return set_error(NSVF_EINVAL, "trilinear_gather_backward_plan: null pointer");
  if (plan_bytes_given < plan_bytes(N, K))
    return set_error(NSVF_EINVAL, "trilinear_gather_backward_plan: plan buffer too small");
  hipStream_t st = as_stream(stream);
  GradWorkspace w;
  // the incidence buffers and sort space do not depend on M or D
  layout(0, N, K, 4, static_cast<char*>(workspace), &w);
  if (workspace_bytes < w.total)
    return set_error(NSVF_EINVAL, "trilinear_gather_backward_plan: workspace too small");
  char* pb = static_cast<char*>(plan);
  return build_plan(feats, N, K, w, reinterpret_cast<int32_t*>(pb),
                    reinterpret_cast<int32_t*>(pb + align256(8 * N * 4)), st);
}

int64_t nsvf_trilinear_gather_backward_workspace(int64_t M, int64_t N, int64_t K, int D,
                                                 void* stream) {
  clear_error();
  if (M < 0 || N <= 0 || K <= 0 || D <= 0) {
    set_error(NSVF_EINVAL, "trilinear_gather_backward_workspace: bad size");
    return -1;
  }
  GradWorkspace w;
  layout(M, N, K, D, nullptr, &w);
  return w.total;
}

int nsvf_trilinear_gather_backward_planned(const int32_t* s_idx, const float* xyz, int64_t M,
                                           const float* centers, const int32_t* feats, int64_t N,
                                           int64_t K, int D, float voxel_size,
                                           const float* grad_out, float* grad_values,
                                           const void* plan, void* workspace,
                                           int64_t workspace_bytes, void* stream) {
  clear_error();
  if (int rc = check_sizes("trilinear_gather_backward", M, N, K, D)) return rc;
  if ((M > 0 && (!s_idx || !xyz || !grad_out)) || !centers || !feats || !grad_values ||
      !workspace)
    return set_error(NSVF_EINVAL, "trilinear_gather_backward: null pointer");
  if ((reinterpret_cast<uintptr_t>(grad_out) | reinterpret_cast<uintptr_t>(grad_values)) & 15)
    return set_error(NSVF_EINVAL, "trilinear_gather_backward: gradients must be 16-byte aligned");
  hipStream_t st = as_stream(stream);
  GradWorkspace w;
  layout(M, N, K, D, static_cast<char*>(workspace), &w);
  if (workspace_bytes < w.total)
    return set_error(NSVF_EINVAL, "trilinear_gather_backward: workspace too small (%lld < %lld)",
                     (long long)workspace_bytes, (long long)w.total);
  // 1. samples sorted by voxel
  sort_by_key(s_idx, M, int32_t(N), w.keys, w.vals, w.keys2, w.vals2, w.counts, st);
  hipLaunchKernelGGL(segment_starts_kernel, dim3(unsigned(ceil_div(N + 1, kBlock))), dim3(kBlock),
                     0, st, w.keys, M, N + 1, w.seg);
  // 2. per-(voxel, corner) partials
  const auto corner = D <= 32   ? voxel_corner_kernel<1>
                      : D <= 64 ? voxel_corner_kernel<2>
                                : voxel_corner_kernel<4>;
  hipLaunchKernelGGL(corner, dim3(unsigned(ceil_div(N, kBlock / 64))), dim3(kBlock), 0, st, w.seg, w.vals, xyz, centers, voxel_size, grad_out, D,
                     N, w.partial);
  // 3. incidences in corner-key order (the plan, or computed here), then
  // one sum per key
  const int32_t* ivals = w.ivals;
  const int32_t* kseg = w.kseg;
  if (plan) {
    ivals = static_cast<const int32_t*>(plan);
    kseg = reinterpret_cast<const int32_t*>(static_cast<const char*>(plan) + align256(8 * N * 4));
  } else if (int rc2 = build_plan(feats, N, K, w, w.ivals, w.kseg, st)) {
    return rc2;
  }
  hipLaunchKernelGGL(key_sum_kernel, dim3(unsigned(ceil_div(K * (D / 4), kBlock))), dim3(kBlock),
                     0, st, kseg, ivals, w.partial, K, D, grad_values);
  return check_launch("trilinear_gather_backward");
}

int nsvf_trilinear_gather_backward(const int32_t* s_idx, const float* xyz, int64_t M,
                                   const float* centers, const int32_t* feats, int64_t N,
                                   int64_t K, int D, float voxel_size, const float* grad_out,
                                   float* grad_values, void* workspace, int64_t workspace_bytes,
                                   void* stream) {
  return nsvf_trilinear_gather_backward_planned(s_idx, xyz, M, centers, feats, N, K, D, voxel_size,
                                                grad_out, grad_values, nullptr, workspace,
                                                workspace_bytes, stream);
}

}  // extern "C"
