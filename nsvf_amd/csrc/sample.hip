// Ray sampling kernels for gfx950: inverse-CDF and uniform.
//
// Op-level kernels keep the `_ext` layout ([B,R,P] bins in, [B,R,S] padded
// samples out; fairnr/clib/src/sample.cpp:23-95).  The row kernel serves the
// Python-level `inverse_cdf_sampling` (fairnr/clib/__init__.py:231-300) in one
// launch: it takes the [N,P] rows directly and derives, for each ray, the
// neighbours the reference's G=200 regrouping and 800-column chunking give it
// (which the trailing-loop quirks read), instead of materialising the
// regrouped chunks.
#include <algorithm>

#include "sample_core.h"

namespace nsvf {
namespace {

constexpr int kSampleBlock = 256;

// Bins of ray j of an op-level [B,R,P] batch buffer.
struct OpBins {
  const int32_t* idx;   // this ray's row
  const float* lo_;
  const float* hi_;
  const float* pr;
  const int32_t* row0;  // first ray of the batch row
  int32_t next;         // slot P of this row in the flat buffer
  __device__ __forceinline__ int32_t id(int k) const { return idx[k]; }
  __device__ __forceinline__ float lo(int k) const { return lo_[k]; }
  __device__ __forceinline__ float hi(int k) const { return hi_[k]; }
  __device__ __forceinline__ float prob(int k) const { return pr[k]; }
  __device__ __forceinline__ int32_t next_first() const { return next; }
  __device__ __forceinline__ int32_t ray0_id(int k) const { return row0[k]; }
};

// Noise read from the flat batch buffer (a read past the row continues into
// the next ray's noise, as the reference's pointer arithmetic does; past the
// end of the buffer it reads 0.5).
struct FlatNoise {
  const float* row;
  int64_t avail;  // readable elements from `row` to the end of the buffer
  __device__ __forceinline__ float at(int k) const { return k < avail ? row[k] : 0.5f; }
};

// Bins of hit ray n of [N,P] rows under the reference's regrouping.
__device__ __forceinline__ void grouped_neighbours(uint32_t n, uint32_t N, uint32_t G,
                                                   uint32_t chunk, int64_t* ray0, int64_t* next) {
  const uint32_t Kc = (N - 1) / G + 1;  // columns per group row (H / G)
  const uint32_t g = n / Kc, c = n - g * Kc;
  const uint32_t c0 = (c / chunk) * chunk;
  const uint32_t W = min(chunk, Kc - c0);
  const uint32_t n0 = g * Kc + c0;
  *ray0 = n0 < N ? n0 : 0;  // rows past N are copies of row 0
  if (c - c0 + 1 >= W && g + 1 >= G) {
    *next = -1;  // one past the chunk buffer
    return;
  }
  // the next column, or the next group row's first of this chunk (64 bits: a
  // group count near 2^31 has rows of one column)
  const int64_t nn = c - c0 + 1 < W ? int64_t(n) + 1 : int64_t(n0) + Kc;
  *next = nn >= int64_t(N) ? 0 : nn;
}

// RowSink that also counts the samples with a voxel id.
struct CountedRowSink {
  RowSink row;
  int valid;
  __device__ __forceinline__ void operator()(int s, int32_t id, float dist, float mid) {
    if (s < row.S && id != -1) ++valid;
    row(s, id, dist, mid);
  }
};

constexpr int kRowWaves = 4;
constexpr int kRowBins = 256;     // bins of a row staged in LDS: 16 KB per block,
constexpr int kWideBins = 1024;   // or 64 KB (two blocks per CU) where rows have more
constexpr int kRowBlocks = 8192;  // more than the chip holds at once

// Rows that a lane walks rather than a wavefront.  A wavefront costs some 0.65
// ns per row however short it is; a lane a walk of its slots, 64 rows side by
// side.  Lane against wavefront, us: 8 slots 16 and 16 for 4,096 rows, 17 and 56
// for 65,536, 151 and 677 for 1,048,576; 16 slots 25 and 16, 31 and 58, 360 and
// 721; 24 slots 33 and 16, 43 and 59, 593 and 782; 32 slots 44 and 17, 55 and 62,
// 897 and 820.  Where dropped samples are counted, a wavefront's rows that might
// drop one run on one of its lanes: 33 slots with noise, 1,048,576 rows, 1,048
// and 1,162.
__host__ inline bool lane_per_row(int64_t rows, int slots, bool count) {
  return slots <= 8 || (slots <= (count ? 40 : 24) && rows >= (1 << 16));
}

__device__ __forceinline__ int first_set(uint64_t mask) {
  return mask ? __ffsll(static_cast<unsigned long long>(mask)) - 1 : 64;
}

// One ray's inverse-CDF samples by a wavefront, into its padded row, with the
// outputs of icdf_ray bit for bit: the same closed-form places as icdf_wave
// (sample_wave.h: step i's sample at i + b_i, bin k's tail at i_k + k, C the
// left-to-right prefix of the probabilities), but every sample is written,
// also one without a voxel id, its distance as it is.  Rows the closed form
// does not cover run icdf_ray on lane 0: no valid first bin or more than
// bins_cap, a negative or NaN probability (C must not fall), a step count or
// size that is not positive and within the row, noise outside [0, 1] (the
// steps' cdf must not fall).  Returns the number of samples written with a
// voxel id; *count: the samples made, *dropped: those that found no slot
// (counted only if kCount, by the walk itself, which stops at a full row).
template <bool kNoise, bool kCount>
__device__ int icdf_row_wave(const OpBins& bins, int P, float steps, float fixed_step,
                             const FlatNoise& noise, int compat, int S, const RowSink& out,
                             int bins_cap, float* C, float* lo, float* hi, int32_t* id,
                             int* count, int* dropped) {
  const int lane = threadIdx.x & 63;
  const auto u_at = [&](int i) { return kNoise ? noise.at(i) : 0.5f; };
  const auto put = [&](int pos, int32_t v, float d, float mid) {
    if (pos < S) {
      out.idx[pos] = v;
      out.dists[pos] = d;
      out.depth[pos] = mid;
    }
  };
  const float ss = fixed_step > 0.0f ? fixed_step : float(1.0 / double(steps));
  const float per = fixed_step > 0.0f ? 1.0f / fixed_step : steps;   // about 1 / ss
  bool seq = !(steps > 0.0f && steps <= float(S) && ss > 0.0f && ss < 1e30f);
  const int T = seq ? 0 : int(ceilf(steps));
  if constexpr (kNoise) {
    for (int i0 = 0; i0 < T; i0 += 64) {
      const int i = i0 + lane;
      const float u = i < T ? noise.at(i) : 0.5f;
      seq = seq || __any(!(u >= 0.0f && u <= 1.0f));
    }
  }
  // bins up to the first without a voxel; their prefix sums (icdf_wave's DPP
  // chain: each sum rounded once, left to right)
  int Pv = 0;
  float c = 0.0f;
  for (int t0 = 0; !seq; t0 += 64) {
    const int k = t0 + lane;
    const int32_t v = k < P ? bins.id(k) : -1;
    const int here = first_set(__ballot(v == -1));
    if (here > 0) {
      if (t0 + here > bins_cap) {
        seq = true;
        break;
      }
      float pk = 0.0f;
      if (lane < here) {
        pk = bins.prob(k);
        lo[k] = bins.lo(k);
        hi[k] = bins.hi(k);
        id[k] = v;
      }
      seq = __any(!(pk >= 0.0f));
      const float q = (lane == 0 && t0 > 0) ? c + pk : pk;
      float run = q;
      for (int i = 1; i < here; ++i) {
        const float left = __int_as_float(__builtin_amdgcn_update_dpp(
            0, __float_as_int(run), 0x138 /* wave_shr:1 */, 0xf, 0xf, false));
        run = left + q;
      }
      c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(run), here - 1));
      if (lane < here) C[k] = run;
    }
    Pv = t0 + here;
    if (here < 64) break;
  }
  wave_sync();
  // T + Pv samples at most, and one past each bin's end in the trailing loop
  if (kCount) seq = seq || int64_t(T) + Pv + P > S;
  if (seq || Pv == 0 || !(c < 1e30f)) {
    int s = 0;
    CountedRowSink sink{out, 0};
    if (lane == 0) {
      if (kNoise)
        s = icdf_ray(bins, P, steps, fixed_step, noise, compat, S, sink);
      else
        s = icdf_ray(bins, P, steps, fixed_step, ConstNoise{0.5f}, compat, S, sink);
    }
    *count = __shfl(s, 0, 64);
    *dropped = __shfl(sink.row.dropped, 0, 64);
    return __shfl(sink.valid, 0, 64);
  }
  int bprev = 0, n = 0, cb = 0;
  float zprev = lo[0], zl = 0.0f, cmax = 0.0f;
  bool done = false;
  for (int base = 0; base < T; base += 64) {
    const int i = base + lane;
    const bool act = i < T;
    int b = Pv;
    float z = 0.0f;
    if (act) {
      const float cdf = (float(i) + u_at(i)) * ss;
      int l = 0, h = Pv;
      while (l < h) {
        const int mid = (l + h) >> 1;
        if (C[mid] < cdf)
          l = mid + 1;
        else
          h = mid;
      }
      b = l;
      if (b < Pv) {
        const float cmin = b > 0 ? C[b - 1] : 0.0f;
        const float u = (cdf - cmin) / (C[b] - cmin);
        z = __fmaf_rn(u, hi[b] - lo[b], lo[b]);
      }
    }
    int bp = __shfl_up(b, 1, 64);
    float zp = __shfl_up(z, 1, 64);
    if (lane == 0) {
      bp = bprev;
      zp = zprev;
    }
    const uint64_t beyond = __ballot(act && b >= Pv);
    const int dl = first_set(beyond);
    if (act && lane < dl) {
      const float zk = b == bp ? zp : lo[b];
      put(i + b, id[b], z - zk, (z + zk) * 0.5f);
    }
    if (beyond) {
      const int bpd = __shfl(bp, dl, 64);
      const float zpd = __shfl(zp, dl, 64);
      done = true;
      n = base + dl + Pv;
      cb = Pv;
      zl = bpd == Pv - 1 ? zpd : lo[Pv - 1];
      cmax = hi[Pv - 1];
      break;
    }
    const int last = min(T - 1 - base, 63);
    bprev = __shfl(b, last, 64);
    zprev = __shfl(z, last, 64);
  }
  // the tails of the crossed bins, a lane per bin
  for (int k0 = 0; k0 < Pv; k0 += 64) {
    const int k = k0 + lane;
    if (k < Pv) {
      const float ck = C[k];
      int ik = int(fminf(fmaxf(floorf(ck * per - 0.5f) + 1.0f, 0.0f), float(T)));
      while (ik > 0 && (float(ik - 1) + u_at(ik - 1)) * ss > ck) --ik;
      while (ik < T && (float(ik) + u_at(ik)) * ss <= ck) ++ik;
      if (ik < T) {
        float zk = lo[k];
        if (ik > 0) {
          const float cdfp = (float(ik - 1) + u_at(ik - 1)) * ss;
          const float cmin = k > 0 ? C[k - 1] : 0.0f;
          if (k == 0 || cdfp > cmin)
            zk = __fmaf_rn((cdfp - cmin) / (ck - cmin), hi[k] - lo[k], lo[k]);
        }
        put(ik + k, id[k], hi[k] - zk, (hi[k] + zk) * 0.5f);
      }
    }
  }
  if (!done) {
    n = T + bprev;
    cb = bprev;
    zl = zprev;
    cmax = hi[cb];
  }
  int valid = min(n, S);
  // trailing tails: bin cb, then bin after bin while the sequential loop goes on
  if (!(done && !compat) && zl < cmax) {
    const int32_t id0 = cb < P ? bins.id(cb) : bins.next_first();
    if (lane == 0) put(n, id0, cmax - zl, (cmax + zl) * 0.5f);
    valid += n < S && id0 != -1;
    ++n;
    for (int base = cb + 1; base < P; base += 64) {
      const int k = base + lane;
      bool ok = false;
      float lk = 0.0f, hk = 0.0f;
      int32_t idk = -1;
      if (k < P) {
        idk = bins.id(k);
        lk = bins.lo(k);
        hk = bins.hi(k);
        ok = (compat ? bins.ray0_id(k) : idk) != -1 && lk < hk;
      }
      const int stop = first_set(__ballot(!ok));
      if (lane < stop) put(n + lane, idk, hk - lk, (hk + lk) * 0.5f);
      valid += __popcll(__ballot(lane < stop && n + lane < S && idk != -1));
      n += stop;
      if (stop < 64) break;
    }
  }
  *count = n;
  *dropped = 0;
  return valid;
}

// A wavefront per row.  kGrouped: [N,P] rows under the reference wrapper's
// regrouping (R unused); otherwise rows of a [B,R,P] batch.  max_valid
// (optional): raised to the largest number of samples with a voxel id in a
// row, which is what the caller trims the rows to.  kCount: flags[1] += dropped
// samples, flags[2] += batch rows whose steps read noise past the buffer.
// Bound: the padded rows' stores (12 S bytes per row) and the serial prefix
// chain of up to 60 sums per row.  A lane per row walked its samples one by
// one, every store to another line: 65,537 rows of up to 60 bins, 778 -> 174 us.
// Rows of few slots keep that form (icdf_lanes_kernel).
template <bool kNoise, bool kGrouped, bool kCount>
__global__ __launch_bounds__(64 * kRowWaves) void icdf_rows_kernel(
    const int32_t* __restrict__ pts_idx, const float* __restrict__ min_depth,
    const float* __restrict__ max_depth, const float* __restrict__ noise,
    const float* __restrict__ probs, const float* __restrict__ steps, int64_t N, int R,
    int P, int S, int G, int chunk, float fixed_step_size, int compat,
    int32_t* __restrict__ out_idx, float* __restrict__ out_depth,
    float* __restrict__ out_dists, int32_t* __restrict__ max_valid,
    unsigned long long* __restrict__ flags, int bins_cap) {
  extern __shared__ float staged[];   // [wave][C, lo, hi, id][bins_cap]
  __shared__ int best;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (threadIdx.x == 0) best = 0;
  __syncthreads();
  float* C = staged + w * 4 * bins_cap;
  float *lo = C + bins_cap, *hi = lo + bins_cap;
  int32_t* id = reinterpret_cast<int32_t*>(hi + bins_cap);
  int most = 0;
  for (int64_t n = int64_t(blockIdx.x) * kRowWaves + w; n < N;
       n += int64_t(gridDim.x) * kRowWaves) {
    int64_t ray0, next;
    if constexpr (kGrouped) {
      grouped_neighbours(uint32_t(n), uint32_t(N), G, chunk, &ray0, &next);
    } else {
      ray0 = n / R * R;
      next = n + 1 < N ? n + 1 : -1;
    }
    const int64_t H = n * P;
    const OpBins bins{pts_idx + H, min_depth + H, max_depth + H, probs + H, pts_idx + ray0 * P,
                      next < 0 ? -1 : pts_idx[next * P]};
    const RowSink row{out_idx + n * S, out_depth + n * S, out_dists + n * S, S, 0};
    const FlatNoise nz{kNoise ? noise + n * S : nullptr, kGrouped ? S : (N - n) * S};
    const float st = steps[n];
    int count, dropped;
    const int valid = icdf_row_wave<kNoise, kCount>(bins, P, st, fixed_step_size, nz, compat, S,
                                                    row, bins_cap, C, lo, hi, id, &count,
                                                    &dropped);
    most = max(most, valid);
    for (int t = min(count, S) + lane; t < S; t += 64) {
      row.idx[t] = -1;
      row.depth[t] = 0.0f;
      row.dists[t] = 0.0f;
    }
    if (kCount && lane == 0) {
      if (dropped) atomicAdd(&flags[1], (unsigned long long)dropped);
      if (!kGrouped && int64_t(int(ceilf(st))) > nz.avail) atomicAdd(&flags[2], 1ull);
    }
    wave_sync();   // the next row's staging must not overtake this row's reads
  }
  if (max_valid) {
    if (lane == 0) atomicMax(&best, most);
    __syncthreads();
    if (threadIdx.x == 0 && best > 0) raise_max(max_valid, best);
  }
}

// A lane per row, each walking its samples: rows of few slots (lane_per_row).
// Arguments as icdf_rows_kernel's.
template <bool kNoise, bool kGrouped, bool kCount>
__global__ __launch_bounds__(kSampleBlock) void icdf_lanes_kernel(
    const int32_t* __restrict__ pts_idx, const float* __restrict__ min_depth,
    const float* __restrict__ max_depth, const float* __restrict__ noise,
    const float* __restrict__ probs, const float* __restrict__ steps, int64_t N, int R,
    int P, int S, int G, int chunk, float fixed_step_size, int compat,
    int32_t* __restrict__ out_idx, float* __restrict__ out_depth,
    float* __restrict__ out_dists, int32_t* __restrict__ max_valid,
    unsigned long long* __restrict__ flags) {
  __shared__ int best;
  if (threadIdx.x == 0) best = 0;
  __syncthreads();
  const int64_t n = int64_t(blockIdx.x) * kSampleBlock + threadIdx.x;
  if (n < N) {
    int64_t ray0, next;
    if constexpr (kGrouped) {
      grouped_neighbours(uint32_t(n), uint32_t(N), G, chunk, &ray0, &next);
    } else {
      ray0 = n / R * R;
      next = n + 1 < N ? n + 1 : -1;
    }
    const int64_t H = n * P;
    const OpBins bins{pts_idx + H, min_depth + H, max_depth + H, probs + H, pts_idx + ray0 * P,
                      next < 0 ? -1 : pts_idx[next * P]};
    CountedRowSink sink{RowSink{out_idx + n * S, out_depth + n * S, out_dists + n * S, S, 0}, 0};
    const FlatNoise nz{kNoise ? noise + n * S : nullptr, kGrouped ? S : (N - n) * S};
    const float st = steps[n];
    int s;
    if (kNoise)
      s = icdf_ray(bins, P, st, fixed_step_size, nz, compat, S, sink);
    else
      s = icdf_ray(bins, P, st, fixed_step_size, ConstNoise{0.5f}, compat, S, sink);
    sink.row.pad_from(min(s, S));
    if (kCount) {
      if (sink.row.dropped) atomicAdd(&flags[1], (unsigned long long)sink.row.dropped);
      if (!kGrouped && int64_t(int(ceilf(st))) > nz.avail) atomicAdd(&flags[2], 1ull);
    }
    if (max_valid && sink.valid > 0) atomicMax(&best, sink.valid);
  }
  if (max_valid) {
    __syncthreads();
    if (threadIdx.x == 0 && best > 0) raise_max(max_valid, best);
  }
}

template <bool kNoise, bool kGrouped>
static void launch_icdf(const int32_t* pts_idx, const float* min_depth, const float* max_depth,
                        const float* noise, const float* probs, const float* steps, int64_t N,
                        int R, int P, int S, int G, int chunk, float fixed_step_size, int compat,
                        int32_t* out_idx, float* out_depth, float* out_dists, int32_t* max_valid,
                        int64_t* flags, void* stream) {
  auto* fl = reinterpret_cast<unsigned long long*>(flags);
  if (lane_per_row(N, S, flags != nullptr)) {
    hipLaunchKernelGGL((flags ? icdf_lanes_kernel<kNoise, kGrouped, true>
                              : icdf_lanes_kernel<kNoise, kGrouped, false>),
                       dim3(unsigned(ceil_div(N, kSampleBlock))), dim3(kSampleBlock), 0,
                       as_stream(stream), pts_idx, min_depth, max_depth, noise, probs, steps, N, R,
                       P, S, G, chunk, fixed_step_size, compat, out_idx, out_depth, out_dists,
                       max_valid, fl);
    return;
  }
  const dim3 grid(unsigned(std::min<int64_t>(ceil_div(N, kRowWaves), kRowBlocks)));
  const int cap = P <= kRowBins ? kRowBins : kWideBins;
  hipLaunchKernelGGL((flags ? icdf_rows_kernel<kNoise, kGrouped, true>
                            : icdf_rows_kernel<kNoise, kGrouped, false>),
                     grid, dim3(64 * kRowWaves), size_t(kRowWaves) * 4 * cap * sizeof(float),
                     as_stream(stream), pts_idx, min_depth,
                     max_depth, noise, probs, steps, N, R, P, S, G, chunk, fixed_step_size, compat,
                     out_idx, out_depth, out_dists, max_valid, fl, cap);
}

// Uniform sampling of one ray (fairnr/clib/src/sample_gpu.cu:42-105) into a
// padded row; the row is first filled as the reference's host wrapper
// allocates it (idx -1, depth 0, dists 0), since the phases read it back.
__global__ __launch_bounds__(kSampleBlock) void uniform_op_kernel(
    const int32_t* __restrict__ pts_idx_all, const float* __restrict__ min_depth_all,
    const float* __restrict__ max_depth_all, const float* __restrict__ noise_all,
    int64_t BR, int P, int S, float step_size, int32_t* __restrict__ out_idx,
    float* __restrict__ out_depth, float* __restrict__ out_dists,
    unsigned long long* __restrict__ flags) {
  const int64_t r = int64_t(blockIdx.x) * kSampleBlock + threadIdx.x;
  if (r >= BR) return;
  const int64_t H = r * P, K = r * S;
  const int32_t* pts_idx = pts_idx_all + H;
  const float* min_depth = min_depth_all + H;
  const float* max_depth = max_depth_all + H;
  const float* noise = noise_all + K;
  int32_t* sidx = out_idx + K;
  float* sdep = out_depth + K;
  float* sdis = out_dists + K;
  for (int t = 0; t < S; ++t) {
    sidx[t] = -1;
    sdep[t] = 0.0f;
    sdis[t] = 0.0f;
  }
  int oob = 0, dropped = 0, stuck = 0;
  int s = 0, ucur = 0, umin = 0, umax = 0;
  float last_min_depth, last_max_depth, curr_depth = 0.0f;
  while (true) {
    if (umax == P || ucur == S || pts_idx[umax] == -1) break;
    // Past S every write is dropped and nothing later reads this phase's
    // counters, so stopping here changes no output and bounds the loop.
    if (s >= S) break;
    last_min_depth = (umin < P) ? min_depth[umin] : 10000.0f;
    last_max_depth = (umax < P) ? max_depth[umax] : 10000.0f;
    if (ucur < S) curr_depth = __fmaf_rn(float(ucur) + noise[ucur], step_size, min_depth[0]);
    if (last_max_depth <= curr_depth && last_max_depth <= last_min_depth) {
      if (s < S) {
        sdep[s] = last_max_depth;
        sidx[s] = pts_idx[umax];
      } else {
        ++dropped;
      }
      umax++;
      s++;
      continue;
    }
    if (curr_depth <= last_min_depth && curr_depth <= last_max_depth) {
      // umin == 0 only when a noise value is exactly 0: the reference then
      // reads the previous ray's last slot (-1 before the buffer start).
      int32_t id;
      if (umin > 0) {
        id = pts_idx[umin - 1];
      } else if (r > 0) {
        id = pts_idx_all[H - 1];
      } else {
        id = -1;
        ++oob;
      }
      if (s < S) {
        sdep[s] = curr_depth;
        sidx[s] = id;
      } else {
        ++dropped;
      }
      ucur++;
      s++;
      continue;
    }
    if (last_min_depth <= curr_depth && last_min_depth <= last_max_depth) {
      if (s < S) {
        sdep[s] = last_min_depth;
        sidx[s] = pts_idx[umin];
      } else {
        ++dropped;
      }
      umin++;
      s++;
      continue;
    }
    ++stuck;  // NaN depths: no branch applies (the reference would spin)
    break;
  }
  int step = 0;
  umin = 0;
  umax = 0;
  for (ucur = 0; ucur < S - 1; ucur++) {
    if (sidx[ucur + 1] == -1) break;
    const float l_depth = sdep[ucur];
    const float r_depth = sdep[ucur + 1];
    sdep[ucur] = (l_depth + r_depth) * 0.5f;
    sdis[ucur] = r_depth - l_depth;
    if (umin < P && sdep[ucur] >= min_depth[umin] && pts_idx[umin] > -1) umin++;
    if (umax < P && sdep[ucur] >= max_depth[umax] && pts_idx[umax] > -1) umax++;
    if (umax == P || pts_idx[umax] == -1) break;
    if (umin - 1 == umax && sdis[ucur] > 0) {
      sdep[step] = sdep[ucur];
      sdis[step] = sdis[ucur];
      sidx[step] = sidx[ucur];
      step++;
    }
  }
  for (int t = step; t < S; t++) sidx[t] = -1;
  if (flags) {
    if (oob) atomicAdd(&flags[0], (unsigned long long)oob);
    if (dropped) atomicAdd(&flags[1], (unsigned long long)dropped);
    if (stuck) atomicAdd(&flags[2], (unsigned long long)stuck);
  }
}

}  // namespace
}  // namespace nsvf

using namespace nsvf;

extern "C" {

int nsvf_inverse_cdf_sampling(const int32_t* pts_idx, const float* min_depth,
                              const float* max_depth, const float* noise,
                              const float* probs, const float* steps, int B,
                              int R, int P, int S, float fixed_step_size,
                              int compat, int32_t* out_idx, float* out_depth,
                              float* out_dists, int64_t* flags, void* stream) {
  clear_error();
  if (B < 0 || R < 0 || P < 0 || S < 0)
    return set_error(NSVF_EINVAL, "inverse_cdf_sampling: negative size");
  const int64_t BR = int64_t(B) * R;
  if (BR == 0 || S == 0) return NSVF_OK;
  if (P == 0) return set_error(NSVF_EINVAL, "inverse_cdf_sampling: no bins (P = 0)");
  if (!pts_idx || !min_depth || !max_depth || !noise || !probs || !steps || !out_idx ||
      !out_depth || !out_dists)
    return set_error(NSVF_EINVAL, "inverse_cdf_sampling: null pointer");
  launch_icdf<true, false>(pts_idx, min_depth, max_depth, noise, probs, steps, BR, R, P, S, 1, 1,
                           fixed_step_size, compat, out_idx, out_depth, out_dists, nullptr, flags,
                           stream);
  return check_launch("inverse_cdf_sampling");
}

static int icdf_rows(const int32_t* pts_idx, const float* min_depth, const float* max_depth,
                     const float* noise, const float* probs, const float* steps, int N, int P,
                     int S, int group, int chunk, float fixed_step_size, int compat,
                     int32_t* out_idx, float* out_depth, float* out_dists, int64_t* flags,
                     int32_t* max_valid, void* stream) {
  clear_error();
  if (N < 0 || P < 0 || S < 0 || group <= 0 || chunk <= 0)
    return set_error(NSVF_EINVAL, "inverse_cdf_sampling_rows: bad size");
  if (N == 0 || S == 0) return NSVF_OK;
  if (P == 0) return set_error(NSVF_EINVAL, "inverse_cdf_sampling_rows: no bins (P = 0)");
  if (!pts_idx || !min_depth || !max_depth || !probs || !steps || !out_idx || !out_depth ||
      !out_dists)
    return set_error(NSVF_EINVAL, "inverse_cdf_sampling_rows: null pointer");
  (noise ? launch_icdf<true, true> : launch_icdf<false, true>)(
      pts_idx, min_depth, max_depth, noise, probs, steps, N, 1, P, S, group, chunk,
      fixed_step_size, compat, out_idx, out_depth, out_dists, max_valid, flags, stream);
  return check_launch("inverse_cdf_sampling_rows");
}

int nsvf_inverse_cdf_sampling_rows(const int32_t* pts_idx, const float* min_depth,
                                   const float* max_depth, const float* noise,
                                   const float* probs, const float* steps, int N,
                                   int P, int S, int group, int chunk,
                                   float fixed_step_size, int compat,
                                   int32_t* out_idx, float* out_depth,
                                   float* out_dists, int64_t* flags, void* stream) {
  return icdf_rows(pts_idx, min_depth, max_depth, noise, probs, steps, N, P, S, group, chunk,
                   fixed_step_size, compat, out_idx, out_depth, out_dists, flags, nullptr, stream);
}

int nsvf_inverse_cdf_sampling_rows_max(const int32_t* pts_idx, const float* min_depth,
                                       const float* max_depth, const float* noise,
                                       const float* probs, const float* steps, int N,
                                       int P, int S, int group, int chunk,
                                       float fixed_step_size, int compat,
                                       int32_t* out_idx, float* out_depth,
                                       float* out_dists, int32_t* max_valid, void* stream) {
  if (!max_valid && N > 0 && S > 0) {
    clear_error();
    return set_error(NSVF_EINVAL, "inverse_cdf_sampling_rows_max: null pointer");
  }
  return icdf_rows(pts_idx, min_depth, max_depth, noise, probs, steps, N, P, S, group, chunk,
                   fixed_step_size, compat, out_idx, out_depth, out_dists, nullptr, max_valid,
                   stream);
}

int nsvf_uniform_ray_sampling(const int32_t* pts_idx, const float* min_depth,
                              const float* max_depth, const float* noise,
                              int B, int R, int P, int S, float step_size,
                              int32_t* out_idx, float* out_depth,
                              float* out_dists, int64_t* flags, void* stream) {
  clear_error();
  if (B < 0 || R < 0 || P < 0 || S < 0)
    return set_error(NSVF_EINVAL, "uniform_ray_sampling: negative size");
  const int64_t BR = int64_t(B) * R;
  if (BR == 0 || S == 0) return NSVF_OK;
  if (P == 0) return set_error(NSVF_EINVAL, "uniform_ray_sampling: no bins (P = 0)");
  if (!pts_idx || !min_depth || !max_depth || !noise || !out_idx || !out_depth || !out_dists)
    return set_error(NSVF_EINVAL, "uniform_ray_sampling: null pointer");
  hipLaunchKernelGGL(uniform_op_kernel, dim3(unsigned(ceil_div(BR, kSampleBlock))),
                     dim3(kSampleBlock), 0, as_stream(stream), pts_idx, min_depth, max_depth, noise,
                     BR, P, S, step_size, out_idx, out_depth, out_dists,
                     reinterpret_cast<unsigned long long*>(flags));
  return check_launch("uniform_ray_sampling");
}

}  // extern "C"
