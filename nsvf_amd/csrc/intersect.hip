// Ray / sparse-voxel intersection kernels for gfx950.
//
// aabb: no tree; a wavefront per ray passes by 64-voxel tiles whose bounding
//       box the ray misses and tests the voxels of the others, one per lane.
// svo:  depth-first traversal of the loose octree, eight lanes per ray (one per
//       child slot), in the reference's visit order (children popped from slot
//       7 down to slot 0); waiting children are kept per tree level in LDS
//       instead of the reference's 256-entry stack in scratch memory.
//
// Semantics follow fairnr/clib/src/intersect_gpu.cu:73-237 and
// intersect.cpp:49-112: first n_max hits per ray, idx -1 padded, depths 0
// padded (the kernels write the pads, so outputs need no pre-fill).
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace nsvf {
namespace {

// ray_aabb of the box of half size h around the centre at c, its three
// coordinates loaded together.
__device__ __forceinline__ bool ray_voxel(const float o[3], const float inv[3], const float* c,
                                          float h, float* lo, float* hi) {
  const float x = c[0], y = c[1], z = c[2];
  const float mn[3] = {x - h, y - h, z - h}, mx[3] = {x + h, y + h, z + h};
  return ray_box(o, inv, mn, mx, lo, hi);
}

// Threads of one launch, at most: HIP takes fewer than 2^32, which batches of
// a ray each (a block of 1,024 threads) or 2^29 octree rays would pass.
constexpr int64_t kLaunchThreads = int64_t(1) << 31;

constexpr int kAabbWaves = 16;
constexpr int kAabbBlock = 64 * kAabbWaves;
constexpr int kAabbTiles = 1024;   // 64-voxel tiles whose boxes a block holds at once
constexpr int kAabbRays = 1024;    // rays per block, at most
constexpr int kAabbAhead = 4;      // tiles a ray's wave loads at once

// Wave-wide minimum of v (not NaN) to lane 63: the running minima of a wave
// scan (DPP: within rows of 16, then row to row).
__device__ __forceinline__ float wave_min63(float v) {
  const auto step = [&v](auto dpp, auto rows) {
    const int o = __builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), dpp(), rows(),
                                              0xF, false);
    v = fminf(v, __int_as_float(o));
  };
  using std::integral_constant;
  step(integral_constant<int, 0x111>{}, integral_constant<int, 0xF>{});  // row_shr:1
  step(integral_constant<int, 0x112>{}, integral_constant<int, 0xF>{});  // row_shr:2
  step(integral_constant<int, 0x114>{}, integral_constant<int, 0xF>{});  // row_shr:4
  step(integral_constant<int, 0x118>{}, integral_constant<int, 0xF>{});  // row_shr:8
  step(integral_constant<int, 0x142>{}, integral_constant<int, 0xA>{});  // row_bcast:15
  step(integral_constant<int, 0x143>{}, integral_constant<int, 0xC>{});  // row_bcast:31
  return v;
}

// Whether a ray can hit any voxel whose centre lies in [mn, mx]: false only
// if ray_aabb is false for every such centre (h >= 0 here).  The rounded
// c - h, c + h, their differences with o and their products with inv are all
// monotone in c, so per axis the box's interval contains every voxel's and
// the running bounds below contain ray_aabb's.  A NaN bound (0 * inf: a
// direction component 0 with the origin on the face, or a NaN input) leaves
// its axis out, as ray_aabb's comparisons with it are false.
__device__ __forceinline__ bool ray_may_hit(const float o[3], const float inv[3],
                                            const float mn[3], const float mx[3], float h) {
  float f_low = 0.0f, f_high = 100000.0f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float t0 = (mn[a] - h - o[a]) * inv[a];
    const float t1 = (mx[a] + h - o[a]) * inv[a];
    if (t0 == t0 && t1 == t1) {
      f_low = fmaxf(f_low, fminf(t0, t1));
      f_high = fminf(f_high, fmaxf(t0, t1));
    }
  }
  return !(f_low > f_high);
}

// One wavefront per ray, the voxels in tiles of 64 consecutive ids.  Each
// block first reduces every tile's centres to a bounding box in LDS; a ray
// then tests 64 tile boxes per step (one per lane) and only the tiles it can
// hit voxel by voxel, a voxel per lane, in id order: the lanes' hits go out at
// the row's count plus the number of hits in lower lanes, so the first n_max
// hits come out in voxel order as in a walk over all voxels.  Voxel ids are
// grid-ordered in every scene here, so a tile is a short piece of a grid line
// or two and a ray passes most by; ids in no order cost a test of every voxel,
// as before, still 64 per step.
// Bound: latency of the tile loads (L2), with 32 waves per CU in flight.
// Against a lane per ray over all voxels (one block per 256 rays, so 8,192
// rays filled an eighth of the chip): 8,192 rays x 6,568 voxels 2,177 us ->
// 45 us (50 with one tile loaded at a time).
__global__ __launch_bounds__(kAabbBlock) void aabb_intersect_kernel(
    const float* __restrict__ ray_start, const float* __restrict__ ray_dir,
    const float* __restrict__ points, int M, int N, int64_t points_bstride,
    int first_block, int blocks_per_batch, int rays_per_block, float half_voxel, int n_max,
    int32_t* __restrict__ idx, float* __restrict__ min_depth,
    float* __restrict__ max_depth) {
  __shared__ float box[6][kAabbTiles];
  __shared__ int32_t counts[kAabbRays];
  const int b = (first_block + blockIdx.x) / blocks_per_batch;
  const int j0 = (first_block + blockIdx.x) % blocks_per_batch * rays_per_block;
  const int rays = min(rays_per_block, M - j0);
  const float* pts = points + b * points_bstride;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const float h_box = fabsf(half_voxel);

  for (int i = threadIdx.x; i < rays; i += kAabbBlock) counts[i] = 0;
  for (int64_t base = 0; base == 0 || base < N; base += 64 * kAabbTiles) {
    const int tiles = int(min(int64_t(kAabbTiles), (N - base + 63) / 64));
    __syncthreads();
    for (int t = wave; t < tiles; t += kAabbWaves) {
      const int64_t k = min(base + 64 * t + lane, int64_t(N) - 1);
      float mn[3], mx[3];
      bool nan = false;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        mn[a] = mx[a] = pts[k * 3 + a];
        nan = nan || mn[a] != mn[a];
      }
      const bool any_nan = __any(nan);  // such a tile is never passed by
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const float lo = wave_min63(mn[a]), hi = -wave_min63(-mx[a]);
        if (lane == 63) {
          box[a][t] = any_nan ? -INFINITY : lo;
          box[3 + a][t] = any_nan ? INFINITY : hi;
        }
      }
    }
    __syncthreads();
    for (int i = wave; i < rays; i += kAabbWaves) {
      const int64_t r = int64_t(b) * M + j0 + i;
      float o[3], inv[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        o[a] = ray_start[r * 3 + a];
        inv[a] = 1.0f / ray_dir[r * 3 + a];
      }
      int cnt = counts[i];
      for (int t0 = 0; t0 < tiles && cnt < n_max; t0 += 64) {
        const int t = t0 + lane;
        bool may = false;
        if (t < tiles) {
          const float mn[3] = {box[0][t], box[1][t], box[2][t]};
          const float mx[3] = {box[3][t], box[4][t], box[5][t]};
          may = ray_may_hit(o, inv, mn, mx, h_box);
        }
        uint64_t todo = __ballot(may);
        while (todo && cnt < n_max) {
          // the next tiles' voxels are loaded together (an absent tile loads
          // the last one again, unused), then tested in order
          int64_t k[kAabbAhead];
          float c[kAabbAhead][3];
          bool have[kAabbAhead];
#pragma unroll
          for (int q = 0; q < kAabbAhead; ++q) {
            have[q] = todo != 0;
            if (have[q]) k[q] = base + 64 * (t0 + __builtin_ctzll(todo)) + lane;
            else k[q] = k[q > 0 ? q - 1 : 0];
            todo &= todo - 1;
            const float* p = pts + min(k[q], int64_t(N) - 1) * 3;
#pragma unroll
            for (int a = 0; a < 3; ++a) c[q][a] = p[a];
          }
#pragma unroll
          for (int q = 0; q < kAabbAhead; ++q) {
            float lo = 0.0f, hi = 0.0f;
            const bool hit =
                have[q] && k[q] < N && ray_voxel(o, inv, c[q], half_voxel, &lo, &hi);
            const uint64_t hits = __ballot(hit);
            const int64_t at = int64_t(cnt) + __popcll(hits & ((1ull << lane) - 1));
            if (hit && at < n_max) {
              idx[r * n_max + at] = int32_t(k[q]);
              min_depth[r * n_max + at] = lo;
              max_depth[r * n_max + at] = hi;
            }
            cnt = int(min(int64_t(cnt) + __popcll(hits), int64_t(n_max)));
          }
        }
      }
      if (base + 64 * kAabbTiles >= N) {  // the last tiles: pad the row
        for (int64_t l = int64_t(cnt) + lane; l < n_max; l += 64) {
          idx[r * n_max + l] = -1;
          min_depth[r * n_max + l] = 0.0f;
          max_depth[r * n_max + l] = 0.0f;
        }
      } else if (lane == 0) {
        counts[i] = cnt;
      }
    }
  }
}

constexpr int kSvoWaves = 4;
constexpr int kSvoBlock = 64 * kSvoWaves;
constexpr int kSvoRays = kSvoBlock / 8;   // rays per block
constexpr int kSvoMaxLevels = 30;
constexpr int kSvoIdBits = 27;            // node ids; the depth sits above them
constexpr uint32_t kSvoLeaf = 31;         // depth code of a waiting leaf

// Half sizes, over the scale, of the boxes an internal node is tested with:
// the reference's loose box, twice the node's octant, or the octant with a
// margin, where svo_check_kernel has found that it holds every leaf below.
constexpr float kSvoLoose = 1.0f, kSvoTight = 0.5f + 0.5f / 64.0f;
constexpr int kSvoChecks = 1024;   // blocks of the check, one flag each
// The check reads the whole tree, 17 us per million nodes, and halves the time
// of a call whose rays hit something.  Where the tree has more than
// kSvoCheckNodes nodes and kSvoCheckPerRay per ray it looks at the rays first:
// if none of kSvoCheckRays of them hits the root's octant, the walk is short
// anyway and the tree passes for one that failed.  On a tree of 4.5 M nodes
// calls of up to 1,024 rays that miss took 24 us without any check, 101 with it
// and 25 so; 64 rays that hit 4,940 us eight children in turn, 376 with the
// loose boxes and 210 so.
constexpr int64_t kSvoCheckNodes = 1 << 18, kSvoCheckPerRay = 64;
constexpr int kSvoCheckRays = 1024;
constexpr int kSvoCheckBlock = 256;

// Whether, for every node of scale s >= 2 and each of its children m, the
// box of half size kSvoTight * s * half_voxel around the node's centre holds
// the child's (a leaf's own box, or the child's of the same form): then it
// holds the boxes of all leaves below, and since a box that holds another is
// hit whenever that is (ray_box is monotone in the box's corners, as rounded),
// a walk that tests these boxes finds the reference's leaves in its order.
// flags[block] = 1 where some child of the block's share is not held; thread
// per (node, slot).  The slack covers the rounding of this test itself.
// rays: kSvoCheckRays or fewer of the call's B_M to look at first (0: none).
__global__ __launch_bounds__(kSvoCheckBlock) void svo_check_kernel(
    const float* __restrict__ centers, const int32_t* __restrict__ children, int T,
    float half_voxel, const float* __restrict__ ray_start, const float* __restrict__ ray_dir,
    int64_t B_M, int rays, int32_t* __restrict__ flags) {
  if (rays > 0) {
    bool hits = false;
    const int root = T - 1;
    const float h = half_voxel * (float(children[int64_t(root) * 9 + 8]) * kSvoTight);
    for (int i = threadIdx.x; i < rays; i += kSvoCheckBlock) {
      const int64_t r = i * B_M / rays;
      float o[3], inv[3], lo, hi;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        o[a] = ray_start[r * 3 + a];
        inv[a] = 1.0f / ray_dir[r * 3 + a];
      }
      hits = hits || ray_voxel(o, inv, centers + int64_t(root) * 3, h, &lo, &hi);
    }
    if (!__syncthreads_or(hits ? 1 : 0)) {
      if (threadIdx.x == 0) flags[blockIdx.x] = 1;
      return;
    }
  }
  bool bad = !(half_voxel > 0.0f);
  const int64_t n = int64_t(T) * 8, stride = int64_t(gridDim.x) * kSvoCheckBlock;
#pragma unroll 2
  for (int64_t i = int64_t(blockIdx.x) * kSvoCheckBlock + threadIdx.x; i < n; i += stride) {
    const int64_t node = i >> 3;
    const int sc = children[node * 9 + 8], c = children[node * 9 + (i & 7)];
    if (sc == 1 || uint32_t(c) >= uint32_t(T)) continue;
    const int csc = children[int64_t(c) * 9 + 8];
    const float own = half_voxel * (float(sc) * kSvoTight);
    const float child = half_voxel * (float(csc) * (csc == 1 ? 1.0f : kSvoTight));
    bad = bad || sc < 2 || csc < 1;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float x = centers[node * 3 + a], y = centers[int64_t(c) * 3 + a];
      const float slack = (fabsf(x) + fabsf(y) + own) * 0x1p-20f;
      bad = bad || !(fabsf(y - x) + child + slack <= own);
    }
  }
  const int any = __syncthreads_or(bad ? 1 : 0);
  if (threadIdx.x == 0) flags[blockIdx.x] = any;
}

// Depth-first traversal, eight lanes per ray: lane s of a ray's group tests
// the child in slot 7 - s of the node being expanded, so an expansion is one
// round of loads (the node's child ids, then the eight children's records and
// centres) and one slab test instead of eight of each in turn, and lane order
// is the visit order: slots 7 down to 0, the order in which the reference
// pops them after pushing 0..7.  Leaves hit before the first internal child
// go out together, at the row's count plus the hits in lower lanes; the
// other hit children wait: their ids and depths in LDS (per stack level and
// lane) and, in bit l of each lane's `pend`, that its child at level l is
// still to visit.  The next node is the first waiting child of the deepest
// level with any.
//
// An internal child with exactly one child of its own stands for that child:
// its lane tests both boxes and goes on with the grandchild, which would be
// visited next and alone.  The reference's octree has a whole level of such
// nodes (voxel centres sit on even half-voxel coordinates, so each finest
// internal node holds one voxel), so most leaves cost no expansion of their
// own.
//
// Guards that keep every ray finite on any input: child ids outside [0,T)
// are skipped, a child is descended into only if its scale is smaller than
// its parent's (so a malformed tree cannot cycle), and at most
// kSvoMaxLevels internal levels are held (a valid tree over int32
// coordinates has at most 31; deeper subtrees are not descended): `depth`
// counts a node's internal ancestors, skipped ones included.
//
// With `flags` (svo_check_kernel's, all 0) internal nodes are tested with
// their octant instead of the reference's box of twice its size: a ray of the
// 100k-voxel cloud's image expands 34 nodes instead of 121, for the same
// leaves.
//
// Bound: VALU issue (82% of cycles with the loose boxes), the dependent loads
// behind it, with up to 20 waves (160 rays) per CU in flight.  A lane per ray
// tested the eight children one after another, each test behind a load of its
// own, with every lane of a wave at another node: 8,192 random rays on the
// 6,568-voxel shell 1,650 us -> 51 us, a 401 x 399 image of 100k
// voxels 4,260 us -> 400 us (128 and 1,080 us with the loose boxes;
// without the skipped links 280 and 1,340 us).
// kShared: one tree for all rays, small enough that 32-bit byte offsets from
// its (uniform) base address every node; else a base per ray and 64 bits.
template <bool kShared>
__global__ __launch_bounds__(kSvoBlock) void svo_intersect_kernel(
    const float* __restrict__ ray_start, const float* __restrict__ ray_dir,
    const float* __restrict__ centers, const int32_t* __restrict__ children,
    int64_t first_ray, int64_t B_M, int M, int T, int64_t centers_bstride,
    int64_t children_bstride, float half_voxel, int n_max, const int32_t* __restrict__ flags,
    int nflags,
    int32_t* __restrict__ idx, float* __restrict__ min_depth, float* __restrict__ max_depth) {
  __shared__ uint32_t waiting_at[kSvoMaxLevels][kSvoBlock];
  // blocks go round the 8 XCDs; each takes one contiguous eighth of the rays,
  // so that the nodes its neighbouring rays share stay in its L2
  const int64_t per_xcd = gridDim.x / 8;
  const int64_t blk = int64_t(blockIdx.x) < per_xcd * 8
                          ? (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3)
                          : int64_t(blockIdx.x);
  const int64_t r = first_ray + blk * kSvoRays + (threadIdx.x >> 3);
  const int s = threadIdx.x & 7;
  const int shift = threadIdx.x & 56;   // this group's first lane in its wave
  const uint32_t before = (1u << s) - 1;
  const bool active = r < B_M;
  const int64_t b = !kShared && active ? r / M : 0;
  const float* cen = kShared ? centers : centers + b * centers_bstride;
  const int32_t* ch = kShared ? children : children + b * children_bstride;
  using Offset = std::conditional_t<kShared, uint32_t, int64_t>;
  // node k's record (child ids, then the scale) and centre
  const auto record = [ch](int k) { return ch + Offset(k) * 9; };
  const auto valid_id = [T](int k) { return uint32_t(k) < uint32_t(T); };
  uint32_t* my_wait = &waiting_at[0][threadIdx.x];
  const uint32_t* group_wait = &waiting_at[0][threadIdx.x & ~7];
  // the group's eight bits of a wave-wide vote
  const auto group_bits = [shift](bool p) { return uint32_t(__ballot(p) >> shift) & 0xFFu; };

  float o[3] = {0.f, 0.f, 0.f}, inv[3] = {0.f, 0.f, 0.f};
  if (active) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      o[a] = ray_start[r * 3 + a];
      inv[a] = 1.0f / ray_dir[r * 3 + a];
    }
  }
  // the box an internal node is tested with
  bool loose = flags == nullptr;
  for (int i = threadIdx.x & 63; i < nflags; i += 64) loose = loose || flags[i] != 0;
  const float box = __any(loose) ? kSvoLoose : kSvoTight;
  const auto test = [&](int k, int scale, float* lo, float* hi) {
    const float h = half_voxel * (float(scale) * (scale == 1 ? 1.0f : box));
    return ray_voxel(o, inv, cen + Offset(k) * 3, h, lo, hi);
  };
  const int64_t row = r * n_max;
  int cnt = 0;
  int node = -1;    // the node to expand (-1: none, the ray is done)
  int level = 0;    // its stack level
  int depth = 0;    // its depth in the tree
  uint32_t pend = 0;
  if (active) {
    const int root = T - 1;
    const int sc = record(root)[8];
    float lo, hi;
    if (test(root, sc, &lo, &hi)) {
      if (sc == 1) {
        if (s == 0) {
          idx[row] = root;
          min_depth[row] = lo;
          max_depth[row] = hi;
        }
        cnt = 1;
      } else {
        node = root;
      }
    }
  }
  while (__any(node >= 0)) {
    bool leaf = false, inner = false;
    int c = -1, cdepth = 0;
    float lo = 0.0f, hi = 0.0f;
    if (node >= 0) {
      int ps = record(node)[8];
      c = record(node)[7 - s];
      cdepth = depth + 1;
      if (valid_id(c)) {
        const int32_t* rec = record(c);
        int sc = rec[8];
        int kids = 0, only = -1;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int k = rec[j];
          kids += valid_id(k);
          only = valid_id(k) ? k : only;
        }
        bool hit = test(c, sc, &lo, &hi);
        if (hit && sc != 1 && sc < ps && cdepth < kSvoMaxLevels && kids == 1) {
          c = only;
          ps = sc;
          sc = record(c)[8];
          ++cdepth;
          hit = test(c, sc, &lo, &hi);
        }
        leaf = hit && sc == 1;
        inner = hit && !leaf && sc < ps && cdepth < kSvoMaxLevels;
      }
    }
    const uint32_t leaves = group_bits(leaf), inners = group_bits(inner);
    // leaves ahead of the first internal child
    const uint32_t first_inner = inners & (0u - inners);
    const uint32_t out = leaves & (first_inner - 1u);
    if (out >> s & 1) {
      const int at = cnt + int(__popc(out & before));
      if (at < n_max) {
        idx[row + at] = c;
        min_depth[row + at] = lo;
        max_depth[row + at] = hi;
      }
    }
    cnt = min(cnt + int(__popc(out)), n_max);
    if (((leaves | inners) & ~out) >> s & 1) {
      my_wait[level * kSvoBlock] = uint32_t(c) | (leaf ? kSvoLeaf : uint32_t(cdepth)) << kSvoIdBits;
      pend |= 1u << level;
    }
    // next: the first waiting child of the deepest level; a waiting leaf goes
    // out here (its test again: the same operands, the same bits)
    uint32_t levels = cnt < n_max ? or8(pend) : 0;
    node = -1;
    wave_sync();
    while (__any(levels != 0 && node < 0)) {
      const bool look = levels != 0 && node < 0;
      const int l = look ? 31 - __clz(int(levels)) : 0;
      const uint32_t waiting = group_bits(look && (pend >> l & 1));
      if (look) {
        const int f = __builtin_ctz(waiting);
        if (s == f) pend &= ~(1u << l);
        if ((waiting & (waiting - 1)) == 0) levels &= ~(1u << l);
        const uint32_t w = group_wait[l * kSvoBlock + f];
        const int k = int(w & ((1u << kSvoIdBits) - 1));
        if (w >> kSvoIdBits != kSvoLeaf) {
          node = k;
          level = l + 1;
          depth = int(w >> kSvoIdBits);
        } else {
          float klo = 0.0f, khi = 0.0f;
          test(k, 1, &klo, &khi);
          if (s == 0) {
            idx[row + cnt] = k;
            min_depth[row + cnt] = klo;
            max_depth[row + cnt] = khi;
          }
          if (++cnt >= n_max) levels = 0;
        }
      }
    }
    wave_sync();
  }
  if (active)
    for (int l = cnt + s; l < n_max; l += 8) {
      idx[row + l] = -1;
      min_depth[row + l] = 0.0f;
      max_depth[row + l] = 0.0f;
    }
}

}  // namespace
}  // namespace nsvf

using namespace nsvf;

extern "C" {

int nsvf_aabb_intersect(const float* ray_start, const float* ray_dir,
                        const float* points, int B, int M, int N,
                        int points_shared, float voxelsize, int n_max,
                        int32_t* idx, float* min_depth, float* max_depth,
                        void* stream) {
  clear_error();
  if (B < 0 || M < 0 || N < 0 || n_max < 0)
    return set_error(NSVF_EINVAL, "aabb_intersect: negative size");
  if (int64_t(B) * M == 0 || n_max == 0) return NSVF_OK;
  if (!ray_start || !ray_dir || !idx || !min_depth || !max_depth || (N > 0 && !points))
    return set_error(NSVF_EINVAL, "aabb_intersect: null pointer");
  // two blocks per CU and batch where the rays allow a ray per wave, so that
  // a block's pass over the voxel centres serves as many rays as it can
  const int64_t rpb =
      std::min<int64_t>(kAabbRays, std::max<int64_t>(kAabbWaves, ceil_div(int64_t(B) * M, 512)));
  const int bpb = int(ceil_div(M, rpb));
  const int64_t blocks = int64_t(bpb) * B;
  if (blocks > INT32_MAX) return set_error(NSVF_EINVAL, "aabb_intersect: too many rays");
  const int64_t pstride = points_shared ? 0 : int64_t(N) * 3;
  for (int64_t first = 0; first < blocks; first += kLaunchThreads / kAabbBlock) {
    const int64_t n = std::min<int64_t>(blocks - first, kLaunchThreads / kAabbBlock);
    hipLaunchKernelGGL(aabb_intersect_kernel, dim3(unsigned(n)), dim3(kAabbBlock), 0,
                       as_stream(stream), ray_start, ray_dir, points, M, N, pstride, int(first),
                       bpb, int(rpb), voxelsize * 0.5f, n_max, idx, min_depth, max_depth);
  }
  return check_launch("aabb_intersect");
}

int64_t nsvf_svo_workspace_bytes(void) { return int64_t(kSvoChecks) * sizeof(int32_t); }

int nsvf_svo_intersect_ws(const float* ray_start, const float* ray_dir,
                          const float* points, const int32_t* children, int B,
                          int M, int T, int tree_shared, float voxelsize,
                          int n_max, int32_t* idx, float* min_depth,
                          float* max_depth, void* workspace,
                          int64_t workspace_bytes, void* stream) {
  clear_error();
  if (B < 0 || M < 0 || T < 0 || n_max < 0)
    return set_error(NSVF_EINVAL, "svo_intersect: negative size");
  if (int64_t(B) * M == 0 || n_max == 0) return NSVF_OK;
  if (T == 0) return set_error(NSVF_EINVAL, "svo_intersect: empty tree");
  if (T >= (1 << kSvoIdBits))
    return set_error(NSVF_EINVAL, "svo_intersect: more than 2^27 nodes");
  if (!ray_start || !ray_dir || !points || !children || !idx || !min_depth || !max_depth)
    return set_error(NSVF_EINVAL, "svo_intersect: null pointer");
  if (workspace && (workspace_bytes < nsvf_svo_workspace_bytes() ||
                    reinterpret_cast<uintptr_t>(workspace) % sizeof(int32_t) != 0))
    return set_error(NSVF_EINVAL, "svo_intersect: workspace too small or misaligned");
  const int64_t BM = int64_t(B) * M;
  const int64_t blocks = ceil_div(BM, kSvoRays);
  if (blocks > INT32_MAX) return set_error(NSVF_EINVAL, "svo_intersect: too many rays");
  const int64_t cstride = tree_shared ? 0 : int64_t(T) * 3;
  const int64_t hstride = tree_shared ? 0 : int64_t(T) * 9;
  hipStream_t st = as_stream(stream);
  int32_t* flags = nullptr;
  int nflags = 0;
  if (workspace && tree_shared) {
    const bool large = T > kSvoCheckNodes + kSvoCheckPerRay * BM;
    const int look = large ? int(std::min<int64_t>(BM, kSvoCheckRays)) : 0;
    flags = static_cast<int32_t*>(workspace);
    nflags = int(std::min<int64_t>(kSvoChecks, ceil_div(int64_t(T) * 8, kSvoCheckBlock)));
    hipLaunchKernelGGL(svo_check_kernel, dim3(unsigned(nflags)), dim3(kSvoCheckBlock), 0, st,
                       points, children, T, voxelsize * 0.5f, ray_start, ray_dir, BM, look, flags);
    if (check_launch("svo_check") != NSVF_OK) return NSVF_ELAUNCH;
  }
  const auto kernel = tree_shared && int64_t(T) * 36 < (int64_t(1) << 32)
                          ? svo_intersect_kernel<true>
                          : svo_intersect_kernel<false>;
  for (int64_t first = 0; first < blocks; first += kLaunchThreads / kSvoBlock) {
    const int64_t n = std::min<int64_t>(blocks - first, kLaunchThreads / kSvoBlock);
    hipLaunchKernelGGL(kernel, dim3(unsigned(n)), dim3(kSvoBlock), 0, st, ray_start, ray_dir,
                       points, children, first * kSvoRays, BM, M, T, cstride, hstride,
                       voxelsize * 0.5f, n_max, flags, nflags, idx, min_depth, max_depth);
  }
  return check_launch("svo_intersect");
}

int nsvf_svo_intersect(const float* ray_start, const float* ray_dir,
                       const float* points, const int32_t* children, int B,
                       int M, int T, int tree_shared, float voxelsize,
                       int n_max, int32_t* idx, float* min_depth,
                       float* max_depth, void* stream) {
  return nsvf_svo_intersect_ws(ray_start, ray_dir, points, children, B, M, T, tree_shared,
                               voxelsize, n_max, idx, min_depth, max_depth, nullptr, 0, stream);
}

}  // extern "C"
