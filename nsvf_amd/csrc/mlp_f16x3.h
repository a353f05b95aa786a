// The FP32 field MLP on the FP16 matrix units, as accurate as on the FP32
// ones (fairnr/modules/field.py:217-279; Linear + ReLU layers and a 4-wide
// head).
//
// An FP32 operand f, scaled by a power of two, is hi + lo with hi = f16(f),
// lo = f16(f - hi): 22 significant bits and the sign of lo.  A product runs
// as Wl Xh + Wh Xl + Wh Xh on v_mfma_f32_16x16x32_f16 with FP32 accumulation
// (Markidis et al., "NVIDIA Tensor Core Programmability, Performance &
// Precision", IPDPSW 2018; Ootomo and Yokota, "Recovering single precision
// accuracy from Tensor Cores while surpassing the FP32 theoretical peak
// performance", IJHPCA 2022), the two small products first, so that only the
// last KT accumulations round at the result's size.  An FP32 MFMA chain of
// K = 128 rounds 32 times; against 64 bits the pruning scores of 6,568 voxels
// are 1.8e-7 off (2-norm) where the FP32 MFMAs' are 2.3e-7.  Three FP16 MFMAs of 16x16x32 take the matrix pipe 48 cycles,
// the eight FP32 16x16x4 MFMAs they replace 256.
//
// FP16 has 5 exponent bits, so every operand is scaled to where its parts are
// normal numbers: a layer's weights by one power of two that brings the
// largest to [2^14, 2^15), a sample's activations by one that does the same
// for its largest (a lane group's 4 x 32 values, reduced across the groups).
// What is smaller than the largest by more than 2^28 keeps an absolute error
// of 2^-39 of it, where FP32 accumulation rounds at 2^-24.  Scaling by powers
// of two is exact and comes back out in the epilogue's fused multiply-add.
//
// A tile with an infinity or NaN in a layer's input (or weights), whose scales
// leave FP32's range, or whose weights one scale does not hold (kF16Spread), is
// reported; the caller then runs it on the
// FP32 MFMAs, so such inputs give what they gave there.
//
// Layout: the field kernels' transposed form Y^T = W X^T.  A wave's tile is
// NT n-tiles of 16 samples; lane (g = lane / 16, c = lane % 16) holds, for
// k-tile kt, features {32 kt + 4 g + i, 32 kt + 16 + 4 g + i} (i < 4) of
// sample c, which are the accumulator rows of m-tiles 2 kt and 2 kt + 1.
// Element i of the FP16 fragment (mt, kt) is the FP32 packing's fragment
// (mt, 8 kt + i) at the same lane, so the FP16 fragments are made from the
// FP32 ones when a block stages its weights in LDS (152 KB for 32 -> 3 x 128
// -> 4, hi and lo: one block of 8 waves per CU; the maxima that choose the scales
// are found on the way).
#pragma once

#include "common.h"

namespace nsvf {

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) float mfma_f32x4;

constexpr int kF16Waves = 8;
constexpr int kF16NT = 2;                 // n-tiles per wave tile
constexpr int kF16Samples = 16 * kF16NT;  // samples per wave tile
// One scale serves a layer whose rows and columns (those that are not 0) have
// maxima of at least this share of the layer's largest weight.  A row or column
// below it, a unit of no weight beside one of much, would be held in fewer bits
// than FP32's: with units 1e7 as large and switched off by their biases, the
// others' gradients were 10% off.  At 2^-10 the errors against 64 bits are
// still the FP32 MFMAs'; layers drawn at random come to 2^-5.
constexpr float kF16Spread = 0x1p-10f;

__device__ __forceinline__ mfma_f32x4 mfma_f16(f16x8 a, f16x8 b, mfma_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// The power of two 2^(141 - e) that scales a value of biased exponent e to
// [2^14, 2^15), and its inverse; e is kept where both are normal numbers.
__device__ __forceinline__ int f16_exponent(float biggest) {
  return max(int(__float_as_uint(biggest) >> 23), 15);
}
__device__ __forceinline__ float f16_scale(int e) { return __int_as_float((268 - e) << 23); }
__device__ __forceinline__ float f16_unscale(int e) { return __int_as_float((e - 14) << 23); }

typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;

// hi and lo parts of s x and t y (powers of two s, t) as packed pairs: the
// products and differences are exact, so each part is rounded once.  One
// v_fma_mix instruction per part (fused in FP32, then rounded to a half of
// the register); written out, since the compiler forms the second hi twice.
__device__ __forceinline__ void f16_split2(float x, float y, float s, float t, f16x2& hi,
                                           f16x2& lo) {
  unsigned int h, l;
  asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(h) : "v"(x), "v"(s));
  asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(h) : "v"(y), "v"(t));
  asm("v_fma_mixlo_f16 %0, %1, %2, -%3 op_sel:[0,0,0] op_sel_hi:[0,0,1]"
      : "=v"(l)
      : "v"(x), "v"(s), "v"(h));
  asm("v_fma_mixhi_f16 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
      : "+v"(l)
      : "v"(y), "v"(t), "v"(h));
  hi = __builtin_bit_cast(f16x2, h);
  lo = __builtin_bit_cast(f16x2, l);
}

// Largest of the 16 lanes of a group, to its lane 15 (DPP row shifts; v >= 0).
__device__ __forceinline__ int row_max15(int v) {
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true));
  return max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true));
}

// Largest of the wave (v >= 0), in a scalar register.
__device__ __forceinline__ int wave_max(int v) {
  const int m = row_max15(v);
  return max(max(__builtin_amdgcn_readlane(m, 15), __builtin_amdgcn_readlane(m, 31)),
             max(__builtin_amdgcn_readlane(m, 47), __builtin_amdgcn_readlane(m, 63)));
}

// Maximum over the four lane groups (lanes c, c + 16, c + 32, c + 48).
__device__ __forceinline__ float groups_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 16, 64));
  return fmaxf(v, __shfl_xor(v, 32, 64));
}

template <int D, int H, int L>
struct F16Mlp {
  static_assert(D % 32 == 0 && H % 32 == 0 && L >= 1, "whole k-tiles");
  static constexpr int KT0 = D / 32, KTH = H / 32, MT = H / 16, NT = kF16NT;
  static constexpr int FRAGS = MT * KT0 + (L - 1) * MT * KTH + KTH;
  static constexpr int BIASES = L * H + 4;
  static constexpr int ROWS = L * H + 4, COLS = D + L * H;  // of all layers
  static constexpr size_t WEIGHT_BYTES = size_t(FRAGS) * 2048;
  // weight fragments, biases, per-layer weight maxima; while staging, those of
  // the rows and columns
  static constexpr size_t LDS_BYTES =
      WEIGHT_BYTES + (BIASES + L + 1 + ROWS + COLS) * sizeof(float);
  static constexpr bool fits() { return H <= 128 && LDS_BYTES <= 160 * 1024; }

  // A block's view of its staged weights.
  const f16x8* w;       // [frag][hi, lo][64 lanes]
  const float* bias;    // hidden layers back to back, then the head's 4
  const float* biggest; // [L + 1] largest |weight| per layer (infinite: no scale)

  static __device__ __forceinline__ int layer_of(int frag) {
    return frag < MT * KT0 ? 0 : min(1 + (frag - MT * KT0) / (MT * KTH), L);
  }

  // Whether a layer has no scale: every tile is for the FP32 units.
  __device__ __forceinline__ bool beyond() const {
    bool out = false;
#pragma unroll
    for (int l = 0; l <= L; ++l) out = out || weight_exponent(l) >= 255;
    return __builtin_amdgcn_readfirstlane(out);
  }

  // Stages the FP32 fragments wfrag (field.pack_mlp's "f32") and biases into
  // lds; every thread of the block calls it.
  static __device__ F16Mlp stage(const float* __restrict__ wfrag,
                                 const float* __restrict__ biases, unsigned char* lds) {
    f16x8* w = reinterpret_cast<f16x8*>(lds);
    float* b = reinterpret_cast<float*>(lds + WEIGHT_BYTES);
    float* big = b + BIASES;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int* rows = reinterpret_cast<int*>(big + L + 1);
    int* cols = rows + ROWS;
    if (threadIdx.x <= L) big[threadIdx.x] = 0.0f;
    for (int i = threadIdx.x; i < ROWS + COLS; i += blockDim.x) rows[i] = 0;
    for (int i = threadIdx.x; i < BIASES; i += blockDim.x) b[i] = biases[i];
    __syncthreads();
    for (int f = wave; f < FRAGS; f += kF16Waves) {
      const int l = layer_of(f), KT = l == 0 ? KT0 : KTH;
      const int n = l == 0 ? f : f - MT * KT0 - (l - 1) * MT * KTH;
      const int g = lane >> 4, c = lane & 15;
      int* col = cols + (l == 0 ? 0 : D + (l - 1) * H) + 32 * (n % KT) + 4 * g;
      int m = 0;  // |x| as integer bits: NaN and infinity are the largest
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int v = __float_as_int(wfrag[(8 * f + i) * 64 + lane]) & 0x7FFFFFFF;
        m = max(m, v);
        const int top = row_max15(v);
        if (c == 15) atomicMax(&col[i < 4 ? i : 12 + i], top);
      }
      m = max(m, __shfl_xor(m, 32, 64));
      m = max(m, __shfl_xor(m, 16, 64));
      if (g == 0 && (l < L || c < 4)) atomicMax(&rows[l * H + 16 * (n / KT) + c], m);
#pragma unroll
      for (int d = 8; d >= 1; d >>= 1) m = max(m, __shfl_xor(m, d, 64));
      if (lane == 0) atomicMax(reinterpret_cast<int*>(big) + l, m);
    }
    __syncthreads();
    unsigned int spread = 0;   // layers with a row or column below kF16Spread
    for (int i = threadIdx.x; i < ROWS + COLS; i += blockDim.x) {
      const int l = i < ROWS ? min(i / H, L) : max(i - ROWS - D + H, 0) / H;
      const float v = __int_as_float(rows[i]);
      if (v != 0.0f && v < big[l] * kF16Spread) spread |= 1u << l;
    }
    __syncthreads();
#pragma unroll
    for (int l = 0; l <= L; ++l)
      if (spread >> l & 1) big[l] = INFINITY;
    __syncthreads();
    for (int f = wave; f < FRAGS; f += kF16Waves) {
      const float s = f16_scale(min(f16_exponent(big[layer_of(f)]), 254));
      f16x8 hi, lo;
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        f16x2 h, l;
        f16_split2(wfrag[(8 * f + i) * 64 + lane], wfrag[(8 * f + i + 1) * 64 + lane], s, s,
                   h, l);
        hi[i] = h[0];
        hi[i + 1] = h[1];
        lo[i] = l[0];
        lo[i + 1] = l[1];
      }
      w[(2 * f) * 64 + lane] = hi;
      w[(2 * f + 1) * 64 + lane] = lo;
    }
    __syncthreads();
    return F16Mlp{w, b, big};
  }

  // The same from FP16 fragments packed before (their scales follow from the
  // layers' largest |weight|, top[0..L]): those of layers 0..L-1 at frags, the
  // head's at head (512 floats per fragment, hi then lo).
  static __device__ F16Mlp stage_packed(const float* __restrict__ frags,
                                        const float* __restrict__ head,
                                        const float* __restrict__ top,
                                        const float* __restrict__ biases, unsigned char* lds) {
    float4* w = reinterpret_cast<float4*>(lds);
    float* b = reinterpret_cast<float*>(lds + WEIGHT_BYTES);
    float* big = b + BIASES;
    constexpr int BODY = (FRAGS - KTH) * 128, ALL = FRAGS * 128;  // float4s
    static_assert(ALL % 512 == 0 && BODY % 512 == 0, "whole rounds of 512 threads");
#pragma unroll 4
    for (int i = threadIdx.x; i < ALL; i += 64 * kF16Waves)
      w[i] = i < BODY ? reinterpret_cast<const float4*>(frags)[i]
                      : reinterpret_cast<const float4*>(head)[i - BODY];
    for (int i = threadIdx.x; i < BIASES; i += 64 * kF16Waves) b[i] = biases[i];
    if (threadIdx.x <= L) big[threadIdx.x] = top[threadIdx.x];
    __syncthreads();
    return F16Mlp{reinterpret_cast<const f16x8*>(w), b, big};
  }

  // What a sample's column carries between layers: the factor that turns a
  // raw accumulator into the layer's sum, and whether the tile must be
  // repeated on the FP32 units.
  struct Column {
    float back[NT];
    bool wild;
  };

  // The scale of a column whose largest |activation| is `biggest` for the
  // layer with weight exponent we; updates col.
  static __device__ __forceinline__ float column_scale(float biggest, int we, int j,
                                                       Column& col) {
    const int e = f16_exponent(biggest);
    const int back = e + we - 282;  // exponent of the accumulator's factor
    col.wild = col.wild || e >= 255 || we >= 255 || back > 120 || (back < -120 && biggest != 0.0f);
    col.back[j] = f16_unscale(e) * f16_unscale(we);
    return f16_scale(min(e, 254));
  }

  __device__ __forceinline__ int weight_exponent(int l) const { return f16_exponent(biggest[l]); }

  // The parts of s x, s y as elements i, i + 1 of an operand.
  static __device__ __forceinline__ void put2(float x, float y, float s, int i, f16x8& oh,
                                              f16x8& ol) {
    f16x2 h, l;
    f16_split2(x, y, s, s, h, l);
    oh[i] = h[0];
    oh[i + 1] = h[1];
    ol[i] = l[0];
    ol[i + 1] = l[1];
  }

  // relu(back sum + bias) of m-tile mt in place, and the columns' running
  // maxima.
  static __device__ __forceinline__ void finish(mfma_f32x4 (&acc)[MT][NT], int mt,
                                                const float* b, int g, const Column& col,
                                                float (&m)[NT]) {
    const float4 bb = *reinterpret_cast<const float4*>(b + 16 * mt + 4 * g);
    const float bv[4] = {bb.x, bb.y, bb.z, bb.w};
#pragma unroll
    for (int j = 0; j < NT; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[mt][j][r] = fmaxf(__fmaf_rn(acc[mt][j][r], col.back[j], bv[r]), 0.0f);
      m[j] = fmaxf(fmaxf(m[j], acc[mt][j][0]), acc[mt][j][1]);
      m[j] = fmaxf(fmaxf(m[j], acc[mt][j][2]), acc[mt][j][3]);
    }
  }

  // The products of MTS m-tiles over KT k-tiles, fragments at A.  Group
  // (mt, kt) issues the small products of k-tile kt of m-tile mt and the
  // large one of m-tile mt - 1, so that four accumulation chains are in
  // flight and every fragment is read two groups (192 matrix cycles) ahead;
  // a scheduling barrier closes the group (left to itself the compiler keeps
  // every m-tile's fragments and accumulators in flight, and spills).
  // finished(mt) runs once acc[mt] is complete, among later products where
  // there are any.
  template <int KT, int MTS, class Finished>
  static __device__ __forceinline__ void products(const f16x8* A, int lane,
                                                  const f16x8 (&xh)[KT][NT],
                                                  const f16x8 (&xl)[KT][NT],
                                                  mfma_f32x4 (&acc)[MTS][NT],
                                                  Finished finished) {
    constexpr int LEAD = 2, NF = MTS * KT, NH = KT + LEAD + 1, NL = LEAD + 1;
    f16x8 h[NH], l[NL];
#pragma unroll
    for (int f = 0; f < LEAD && f < NF; ++f) {
      h[f % NH] = A[(2 * f) * 64 + lane];
      l[f % NL] = A[(2 * f + 1) * 64 + lane];
    }
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int mt = 0; mt <= MTS; ++mt) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        const int f = mt * KT + kt, n = f + LEAD;
        if (n < NF) {
          h[n % NH] = A[(2 * n) * 64 + lane];
          l[n % NL] = A[(2 * n + 1) * 64 + lane];
        }
        if (mt < MTS) {
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acc[mt][j] = mfma_f16(l[f % NL], xh[kt][j],
                                  kt == 0 ? mfma_f32x4{0.f, 0.f, 0.f, 0.f} : acc[mt][j]);
        }
        if (mt > 0) {
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acc[mt - 1][j] = mfma_f16(h[(f - KT) % NH], xh[kt][j], acc[mt - 1][j]);
        }
        if (mt < MTS) {
#pragma unroll
          for (int j = 0; j < NT; ++j) acc[mt][j] = mfma_f16(h[f % NH], xl[kt][j], acc[mt][j]);
        }
        if (kt == 0 && mt > 1) finished(mt - 2);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
    finished(MTS - 1);
  }

  // One layer: the sums, finished among the products, then the next layer's
  // operands: each column scaled by its own maximum for the weight exponent
  // we.
  template <int KT>
  static __device__ __forceinline__ void layer(const f16x8* A, const float* b, int lane, int g,
                                               int we, Column& col, const f16x8 (&xh)[KT][NT],
                                               const f16x8 (&xl)[KT][NT], f16x8 (&oh)[KTH][NT],
                                               f16x8 (&ol)[KTH][NT]) {
    mfma_f32x4 acc[MT][NT];
    float m[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) m[j] = 0.0f;
    products<KT, MT>(A, lane, xh, xl, acc,
                     [&](int mt) { finish(acc, mt, b, g, col, m); });
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const float s = column_scale(groups_max(m[j]), we, j, col);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 4; r += 2)
          put2(acc[mt][j][r], acc[mt][j][r + 1], s, 4 * (mt & 1) + r, oh[mt >> 1][j],
               ol[mt >> 1][j]);
    }
  }

  // One wave tile: x[j][8 kt + i] = this lane's input features of n-tile j in
  // k-tile order; out[j] = the head's 4 sums (biases added) of sample c on
  // the lanes of group 0.  hook(l) runs after layer l = 0 and 1 (a caller's
  // loads for its next tile).  False: repeat the tile on the FP32 units.
  template <class Hook>
  __device__ __forceinline__ bool tile(const float (&x)[NT][D / 4], int lane, int g,
                                       mfma_f32x4 (&out)[NT], Hook hook) const {
    Column col;
    col.wild = false;
    f16x8 xh[KTH][NT], xl[KTH][NT];
    {
      f16x8 x0h[KT0][NT], x0l[KT0][NT];
      const int we = weight_exponent(0);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        int m = 0;
#pragma unroll
        for (int k = 0; k < D / 4; ++k) m = max(m, __float_as_int(x[j][k]) & 0x7FFFFFFF);
        m = max(m, __shfl_xor(m, 16, 64));
        m = max(m, __shfl_xor(m, 32, 64));
        const float s = column_scale(__int_as_float(m), we, j, col);
#pragma unroll
        for (int k = 0; k < D / 4; k += 2)
          put2(x[j][k], x[j][k + 1], s, k & 7, x0h[k >> 3][j], x0l[k >> 3][j]);
      }
      layer<KT0>(w, bias, lane, g, weight_exponent(1), col, x0h, x0l, xh, xl);
    }
    hook(0);
#pragma unroll 1
    for (int l = 1; l < L; ++l) {
      layer<KTH>(w + 2 * (MT * KT0 + (l - 1) * MT * KTH) * 64, bias + l * H, lane, g,
                 weight_exponent(l + 1), col, xh, xl, xh, xl);
      if (l == 1) hook(1);
    }
    {
      mfma_f32x4 head[1][NT];
      products<KTH, 1>(w + 2 * (FRAGS - KTH) * 64, lane, xh, xl, head, [](int) {});
#pragma unroll
      for (int j = 0; j < NT; ++j) out[j] = head[0][j];
    }
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        out[j][r] = __fmaf_rn(out[j][r], col.back[j], bias[L * H + r]);
    return !__any(col.wild);
  }
};

}  // namespace nsvf
