// Shared helpers for the gfx950 kernels and their C-ABI launchers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>

#include "../../include/nsvf_amd.h"

namespace nsvf {

// Sentinel depth of padded hit slots and samples (fairnr/clib/__init__.py:36).
constexpr float kMaxDepth = 10000.0f;

// Records the error text for nsvf_last_error() and returns `code`.
int set_error(int code, const char* fmt, ...);
void clear_error();

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// Checks the launch that was just enqueued.
inline int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return set_error(NSVF_ELAUNCH, "%s: %s", what, hipGetErrorString(e));
  return NSVF_OK;
}

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// atomicMax for a maximum that thousands of blocks raise: atomics on one
// address go one after another, so those that would change nothing are left
// out (a stale value read here only costs the atomic).
__device__ __forceinline__ void raise_max(int32_t* p, int32_t v) {
  if (v > __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(p, v);
}

// Bitwise or of v over each group of 8 lanes, to all of them (DPP: lane ^ 1,
// lane ^ 2, then the mirror of the 8).
__device__ __forceinline__ uint32_t or8(uint32_t v) {
  v |= uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0xB1, 0xF, 0xF, true));
  v |= uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x4E, 0xF, 0xF, true));
  v |= uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x141, 0xF, 0xF, true));
  return v;
}

// Makes this wavefront's earlier LDS writes visible to all its lanes (a
// barrier for one wave; waves of a block do not wait for each other).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Slab test of one ray against one axis-aligned box (fairnr/clib/src/
// intersect_gpu.cu:73-122): the same comparisons and ternaries, so an axis
// whose bounds come out NaN (direction 0 and origin on the slab plane) fails
// every comparison and is skipped.  `inv` holds IEEE reciprocals of the
// direction, computed once per ray.  Built with -ffp-contract=off, so every
// product and difference below is rounded on its own.
__device__ __forceinline__ bool ray_aabb(const float o[3], const float inv[3],
                                         float cx, float cy, float cz, float h,
                                         float* out_lo, float* out_hi) {
  float f_low = 0.0f;
  float f_high = 100000.0f;
  const float c[3] = {cx, cy, cz};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    float lo = (c[a] - h - o[a]) * inv[a];
    float hi = (c[a] + h - o[a]) * inv[a];
    if (hi < lo) {
      float t = lo;
      lo = hi;
      hi = t;
    }
    if (hi < f_low) return false;
    if (lo > f_high) return false;
    f_low = (lo > f_low) ? lo : f_low;
    f_high = (hi < f_high) ? hi : f_high;
    if (f_low > f_high) return false;
  }
  *out_lo = f_low;
  *out_hi = f_high;
  return true;
}

// Slab test against a box given by its corners; with mn = fp32(c - h) and
// mx = fp32(c + h) this is the reference's test (intersect_gpu.cu:93-94
// evaluates (c - h) - o and (c + h) - o) bit for bit.  The reference returns
// early (per axis: hi < f_low, lo > f_high, then f_low > f_high); here every
// axis runs and only the final f_low > f_high decides, which is the same
// test: f_low only grows and f_high only shrinks, so any early exit leaves
// f_low > f_high at the end, and without one the running values are the
// reference's.  The swap is a compare-and-select, as the reference's
// ternaries, so an axis whose bounds come out NaN (direction 0 and origin on
// the slab plane) is not swapped (a min / max pair would drop its NaN).  The
// running bounds then ignore a NaN as the reference's failed comparisons do:
// fmaxf returns the other operand, and the exit depth is a compare-and-select
// again, since fminf takes -0 for less than +0, the reference's comparison does
// not, and an exit depth of 0 keeps the sign of the first axis (0.5% of the
// traversals' time).  No branches: the traversals
// run one test per child and lane without divergence, and the three axes'
// loads are in flight together.
__device__ __forceinline__ bool ray_box(const float o[3], const float inv[3], const float mn[3],
                                        const float mx[3], float* out_lo, float* out_hi) {
  float f_low = 0.0f;
  float f_high = 100000.0f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float l0 = (mn[a] - o[a]) * inv[a];
    const float h0 = (mx[a] - o[a]) * inv[a];
    const bool sw = h0 < l0;
    const float lo = sw ? h0 : l0;
    const float hi = sw ? l0 : h0;
    f_low = fmaxf(f_low, lo);
    f_high = hi < f_high ? hi : f_high;
  }
  *out_lo = f_low;
  *out_hi = f_high;
  return !(f_low > f_high);
}

}  // namespace nsvf
