// Device-wide exclusive prefix sum of int32 counts: a launch for the tiles'
// sums and one for the scans within the tiles, where each block adds up the
// sums before its own (more than kDirectTiles tiles have theirs scanned by one
// workgroup in between).  The calls are short chains of launches of about 4.6
// us each with nothing beside them, so launches are what they cost: the
// workgroup in between alone took 6.5 us for 27,200 counts and 13.5 for
// 160,000.  Used to turn per-ray hit flags into compacted ray ranks and per-ray sample
// counts into sample-stream offsets, without a host round trip.
#include <algorithm>

#include "common.h"

namespace nsvf {
namespace {

constexpr int kScanBlock = 256;
constexpr int kScanItems = 8;                      // per thread
constexpr int kScanTile = kScanBlock * kScanItems;  // elements per block
constexpr int kPartialItems = 64;                 // per thread, block-sum pass
constexpr int kMaxPartials = kScanBlock * kPartialItems;
constexpr int kDirectTiles = 4096;  // 16 loads per thread in the last block

__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(v, d, 64);
    if (lane >= d) v += u;
  }
  return v;
}

// Inclusive scan of one value per thread across the workgroup.
__device__ __forceinline__ int block_incl_scan(int v, int* smem) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = wave_incl_scan(v);
  if (lane == 63) smem[wave] = v;
  __syncthreads();
  int add = 0;
  for (int w = 0; w < wave; ++w) add += smem[w];
  __syncthreads();
  return v + add;
}

// Sum over the workgroup, in every thread.
__device__ __forceinline__ int block_sum(int v, int* smem) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  if ((threadIdx.x & 63) == 0) smem[threadIdx.x >> 6] = v;
  __syncthreads();
  int sum = 0;
#pragma unroll
  for (int w = 0; w < kScanBlock / 64; ++w) sum += smem[w];
  __syncthreads();
  return sum;
}

// The sums of the tiles before this block's.
__device__ __forceinline__ int tiles_before(const int32_t* __restrict__ partial, int* smem) {
  int s = 0;
  for (unsigned i = threadIdx.x; i < blockIdx.x; i += kScanBlock) s += partial[i];
  return block_sum(s, smem);
}

__device__ __forceinline__ int load_tile(const int32_t* __restrict__ in, int64_t base, int64_t n,
                                         int v[kScanItems]) {
  int s = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    v[i] = base + i < n ? in[base + i] : 0;
    s += v[i];
  }
  return s;
}

__global__ __launch_bounds__(kScanBlock) void scan_reduce_kernel(const int32_t* __restrict__ in,
                                                                 int64_t n,
                                                                 int32_t* __restrict__ partial) {
  __shared__ int smem[kScanBlock / 64];
  int v[kScanItems];
  const int s = block_sum(
      load_tile(in, int64_t(blockIdx.x) * kScanTile + threadIdx.x * kScanItems, n, v), smem);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// One workgroup scans up to kMaxPartials block sums (exclusive, in place) and
// writes the grand total.
__global__ __launch_bounds__(kScanBlock) void scan_partials_kernel(int32_t* __restrict__ partial,
                                                                   int nb,
                                                                   int32_t* __restrict__ total) {
  __shared__ int smem[kScanBlock / 64];
  const int base = threadIdx.x * kPartialItems;
  int s = 0;
  for (int i = 0; i < kPartialItems; ++i)
    if (base + i < nb) s += partial[base + i];
  const int incl = block_incl_scan(s, smem);
  int run = incl - s;
  for (int i = 0; i < kPartialItems; ++i) {
    if (base + i < nb) {
      const int v = partial[base + i];
      partial[base + i] = run;
      run += v;
    }
  }
  if (threadIdx.x == kScanBlock - 1 && total) *total = incl;
}

// kDirect: partial holds the tiles' sums, and the last block writes the total;
// otherwise their exclusive scan.
template <bool kDirect>
__global__ __launch_bounds__(kScanBlock) void scan_apply_kernel(const int32_t* in, int64_t n,
                                                                const int32_t* __restrict__ partial,
                                                                int32_t* out,
                                                                int32_t* __restrict__ total) {
  __shared__ int smem[kScanBlock / 64];
  const int64_t base = int64_t(blockIdx.x) * kScanTile + threadIdx.x * kScanItems;
  int v[kScanItems];
  const int s = load_tile(in, base, n, v);
  const int before = kDirect ? tiles_before(partial, smem) : partial[blockIdx.x];
  const int incl = block_incl_scan(s, smem);
  int run = before + incl - s;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    if (base + i < n) out[base + i] = run;
    run += v[i];
  }
  if (kDirect && total && blockIdx.x == gridDim.x - 1 && threadIdx.x == kScanBlock - 1)
    *total = run;
}

// The two scans between a view's traversal and its samplers, and what goes
// with them: partial[0, tiles) the hit rays and partial[tiles, 2 tiles) the
// slots of each tile of rays, and zero cleared to 0 ...
__global__ __launch_bounds__(kScanBlock) void offsets_reduce_kernel(
    const int32_t* __restrict__ flag, const int32_t* __restrict__ bound, int64_t R,
    int32_t* __restrict__ partial, int32_t* __restrict__ zero) {
  __shared__ int smem[kScanBlock / 64];
  const int64_t base = int64_t(blockIdx.x) * kScanTile + threadIdx.x * kScanItems;
  int v[kScanItems];
  const int hits = block_sum(load_tile(flag, base, R, v), smem);
  const int slots = block_sum(load_tile(bound, base, R, v), smem);
#pragma unroll
  for (int i = 0; i < kScanItems; ++i)
    if (base + i < R) zero[base + i] = 0;
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = hits;
    partial[gridDim.x + blockIdx.x] = slots;
  }
}

// ... then every ray's rank among the hit rays, the list of these, and every
// ray's slot offset; scalars = {hit rays, slots, 0, ...}.  kDirect: as
// scan_apply_kernel's, for both halves of partial.
template <bool kDirect>
__global__ __launch_bounds__(kScanBlock) void offsets_apply_kernel(
    const int32_t* __restrict__ flag, const int32_t* __restrict__ bound, int64_t R,
    const int32_t* __restrict__ partial, int32_t* __restrict__ rank, int32_t* __restrict__ list,
    int32_t* __restrict__ off, int32_t* __restrict__ scalars, int nscalars) {
  __shared__ int smem[kScanBlock / 64];
  const int64_t base = int64_t(blockIdx.x) * kScanTile + threadIdx.x * kScanItems;
  int f[kScanItems], v[kScanItems];
  const int sf = load_tile(flag, base, R, f);
  const int sv = load_tile(bound, base, R, v);
  const int32_t* slots = partial + gridDim.x;
  int hit = (kDirect ? tiles_before(partial, smem) : partial[blockIdx.x]) +
            block_incl_scan(sf, smem) - sf;
  int slot = (kDirect ? tiles_before(slots, smem) : slots[blockIdx.x]) +
             block_incl_scan(sv, smem) - sv;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    if (base + i < R) {
      rank[base + i] = hit;
      off[base + i] = slot;
      if (f[i]) list[hit] = int32_t(base + i);
    }
    hit += f[i];
    slot += v[i];
  }
  if (blockIdx.x == gridDim.x - 1) {
    if (threadIdx.x >= 2 && int(threadIdx.x) < nscalars) scalars[threadIdx.x] = 0;
    if (threadIdx.x == kScanBlock - 1) {
      scalars[0] = hit;
      scalars[1] = slot;
    }
  }
}

}  // namespace

// Exclusive scan of n int32 values into `out` (may alias `in`), grand total
// into *total (device).  `partial` needs scan_partials_size(n) ints.
int scan_exclusive_i32(const int32_t* in, int32_t* out, int64_t n, int32_t* partial,
                       int32_t* total, hipStream_t stream) {
  if (n < 0) return set_error(NSVF_EINVAL, "scan: negative n");
  const int64_t nb = ceil_div(n, kScanTile);
  if (nb > kMaxPartials) return set_error(NSVF_EINVAL, "scan: n too large (%lld)", (long long)n);
  if (n == 0) {
    hipLaunchKernelGGL(scan_partials_kernel, dim3(1), dim3(kScanBlock), 0, stream, partial, 0,
                       total);
    return check_launch("scan");
  }
  hipLaunchKernelGGL(scan_reduce_kernel, dim3(unsigned(nb)), dim3(kScanBlock), 0, stream, in, n,
                     partial);
  const bool direct = nb <= kDirectTiles;
  if (!direct)
    hipLaunchKernelGGL(scan_partials_kernel, dim3(1), dim3(kScanBlock), 0, stream, partial,
                       int(nb), total);
  hipLaunchKernelGGL(direct ? scan_apply_kernel<true> : scan_apply_kernel<false>,
                     dim3(unsigned(nb)), dim3(kScanBlock), 0, stream, in, n, partial, out, total);
  return check_launch("scan");
}

int64_t scan_partials_size(int64_t n) { return ceil_div(n, kScanTile) + 1; }

}  // namespace nsvf

extern "C" {

int64_t nsvf_scan_workspace_ints(int64_t n) { return nsvf::scan_partials_size(n); }

int nsvf_scan_exclusive_i32(const int32_t* in, int32_t* out, int64_t n,
                            int32_t* workspace, int32_t* total, void* stream) {
  nsvf::clear_error();
  if ((n > 0 && (!in || !out)) || !workspace)
    return nsvf::set_error(NSVF_EINVAL, "scan_exclusive_i32: null pointer");
  return nsvf::scan_exclusive_i32(in, out, n, workspace, total, nsvf::as_stream(stream));
}

int64_t nsvf_render_offsets_workspace_ints(int64_t R) {
  return 2 * nsvf::ceil_div(R, nsvf::kScanTile);
}

int nsvf_render_offsets(const int32_t* hit_flag, const int32_t* bound, int64_t R, int32_t* rank,
                        int32_t* list, int32_t* off, int32_t* zero, int32_t* scalars,
                        int nscalars, int32_t* workspace, void* stream) {
  using namespace nsvf;
  clear_error();
  if (R < 0 || nscalars < 2 || nscalars > kScanBlock)
    return set_error(NSVF_EINVAL, "render_offsets: bad size");
  if (!scalars || (R > 0 && (!hit_flag || !bound || !rank || !list || !off || !zero || !workspace)))
    return set_error(NSVF_EINVAL, "render_offsets: null pointer");
  const int64_t tiles = ceil_div(R, kScanTile);
  if (tiles > kMaxPartials)
    return set_error(NSVF_EINVAL, "render_offsets: too many rays (%lld)", (long long)R);
  const dim3 grid(unsigned(std::max<int64_t>(tiles, 1)));
  hipStream_t st = as_stream(stream);
  if (R > 0)
    hipLaunchKernelGGL(offsets_reduce_kernel, grid, dim3(kScanBlock), 0, st, hit_flag, bound, R,
                       workspace, zero);
  const bool direct = tiles <= kDirectTiles;
  for (int k = 0; k < 2 && !direct; ++k)
    hipLaunchKernelGGL(scan_partials_kernel, dim3(1), dim3(kScanBlock), 0, st,
                       workspace + k * tiles, int(tiles), nullptr);
  hipLaunchKernelGGL(direct ? offsets_apply_kernel<true> : offsets_apply_kernel<false>, grid,
                     dim3(kScanBlock), 0, st, hit_flag, bound, R, workspace, rank, list, off,
                     scalars, nscalars);
  return check_launch("render_offsets");
}

}  // extern "C"
