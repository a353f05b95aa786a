// The field MLP for training, the differentiable counterpart of
// fairnr/modules/field.py:217-279 (Linear + ReLU layers, then sigma and
// sigmoid RGB) that the reference trains through torch autograd: forward and
// backward on the 16-bit matrix units (mlp_f16x3.h and
// mlp_train_backward_kernel below), and on v_mfma_f32_16x16x4_f32 (FP32
// operands, FP32 accumulation) where those do not reach.  First the latter.
//
// Layout.  As in the field kernels, a layer runs transposed, Y^T = W X^T:
// weight fragments are operand A (rows = output features), activations
// operand B (columns = the wave's 16 samples).  Lane (g = lane / 16,
// c = lane % 16) holds, for k-tile 4t + i, feature 16t + 4g + i of sample c,
// and a layer's accumulator for m-tile mt holds features 16mt + 4g + r in
// its four registers -- the operand order of the next layer's k-tiles, so
// activations stay in registers through all layers.  The backward products
// dX^T = W^T dY^T use fragments of W^T packed in the same order.
//
// FP32 backward kernel.  A block of 8 waves takes 128 samples at a time (16 per
// wave).  Each wave recomputes its tile's forward pass (every layer's output
// kept in registers), then walks the layers back: the head's dlogits (the
// sigmoid's derivative fused), then per layer dz = dh * (h > 0), the input
// gradient dh_prev = W^T dz and the weight gradient dW = dz^T h_prev.  The
// weight gradient sums over samples, which sit in the wrong operand position
// (across the accumulator's columns); so each wave writes its tile's dz and
// h_prev to LDS, and after a barrier every wave accumulates its own rows of
// dW (one m-tile of each hidden layer, one column tile of the head) over the
// block's 128 samples, 4 samples per MFMA step, with a column of ones for the
// bias gradient.  These accumulators stay in registers for the whole kernel;
// at the end each block writes its partial sums, and a second kernel adds
// the blocks' partials in block order.  The sums therefore run in a fixed
// order for a given sample count: the gradients are deterministic, with no
// atomics.
//
// That is the FP32 kernel, which runs for the samples beside an input that is
// not finite (or far outside FP16's reach) only; the others run on FP16 parts at
// FP32 accuracy, and the split-BF16 form (FieldMLPx3) is the same backward
// kernel on BF16 parts: an FP32 operand f is hi + lo with hi = bf16(f), lo =
// bf16(f - hi), a product Wl Xh + Wh Xl + Wh Xh in FP32 accumulators.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "mlp_f16x3.h"

namespace nsvf {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int kTrainWaves = 8;
constexpr int kTrainBlock = 64 * kTrainWaves;
constexpr int kTrainChunk = 16 * kTrainWaves;  // samples per block step
constexpr int kBwdChunk = 64;                  // of the 16-bit backward kernel
static_assert(kTrainChunk == 2 * kBwdChunk, "the FP32 kernel's steps are two of its chunks");
constexpr int kLdsRow = 144;  // floats per LDS row: 144 = 16 mod 64 banks
constexpr int kMaxTrainBlocks = 256;

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

// (a, b) as packed bf16 pairs hi = bf16(a, b) and lo = bf16(a - hi, b - hi)
// (round to nearest even; the differences are exact in FP32).
__device__ __forceinline__ void split2(float a, float b, unsigned int& hi, unsigned int& lo) {
  const bf16x2 h = __builtin_convertvector(f32x2{a, b}, bf16x2);
  const f32x2 hf = __builtin_convertvector(h, f32x2);
  const bf16x2 l = __builtin_convertvector(f32x2{a - hf[0], b - hf[1]}, bf16x2);
  hi = __builtin_bit_cast(unsigned int, h);
  lo = __builtin_bit_cast(unsigned int, l);
}

// Closes one m-tile's loads and MFMAs: left to itself the scheduler hoists
// the weight loads of every later m-tile (they depend on nothing) and runs
// out of registers.
__device__ __forceinline__ void tile_fence() { __builtin_amdgcn_sched_barrier(0); }

// The weights' address as a value the compiler cannot see through: the
// weight loads of a tile loop are loop-invariant, and hoisted out of it they
// would need hundreds of registers.
template <class P>
__device__ __forceinline__ P opaque(P p) {
  asm volatile("" : "+s"(p));
  return p;
}

// acc += sum over k-tiles kt of A[kt * 64 + lane] x[kt]: the fragment loads go
// at most 8 ahead of their MFMAs (a fence every 8 k-tiles).
template <int KT>
__device__ __forceinline__ f32x4 mfma_chain(const float* __restrict__ A, const float (&x)[KT],
                                            int lane) {
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) {
    acc = mfma4(A[kt * 64 + lane], x[kt], acc);
    if (kt % 8 == 7) tile_fence();
  }
  return acc;
}

// The logistic function, 1 / (1 + e^-x), in IEEE single precision.
__device__ __forceinline__ float logistic(float x) { return 1.0f / (1.0f + expf(-x)); }

// Offsets (in 64-float fragments) of the packed weights of an MLP with input
// width D, L hidden layers of width H and a 4-wide head.
template <int D, int H, int L>
struct TrainDims {
  static constexpr int KT0 = D / 4, KTH = H / 4, MT = H / 16, MT0 = D / 16;
  // forward fragments: layer 0 [MT][KT0], layers 1..L-1 [MT][KTH], head [KTH]
  static constexpr int F_HIDDEN = MT * KT0;  // first fragment of layer 1
  static constexpr int F_HEAD = MT * KT0 + (L - 1) * MT * KTH;
  static constexpr int F_FRAGS = F_HEAD + KTH;
  // transposed fragments: layer 0 [MT0][KTH], layers 1..L-1 [MT][KTH], head [MT]
  static constexpr int T_HIDDEN = MT0 * KTH;
  static constexpr int T_HEAD = MT0 * KTH + (L - 1) * MT * KTH;
  static constexpr int T_FRAGS = T_HEAD + MT;
  static constexpr int64_t T_BASE = int64_t(F_FRAGS) * 64;
  static constexpr int64_t BIAS_BASE = T_BASE + int64_t(T_FRAGS) * 64;
  // per layer: largest |w|, largest row sum |w|, largest column sum |w|,
  // largest b (0 at least) (L + 1 of each)
  static constexpr int64_t STATS_BASE = BIAS_BASE + int64_t(L) * H + 4;
  // parameter gradients in torch order: W_0 [H][D], b_0 [H], ..., W_L [4][H], b_L [4]
  static constexpr int64_t P_W0 = 0, P_B0 = int64_t(H) * D;
  static constexpr int64_t P_LAYER1 = P_B0 + H;
  static constexpr int64_t P_HEAD = P_LAYER1 + int64_t(L - 1) * (int64_t(H) * H + H);
  static constexpr int64_t PARAMS = P_HEAD + 4 * H + 4;
  // split-BF16 fragments (1024 bf16 each: 512 hi, 512 lo), 32-wide k-tiles:
  // layer 0 [MT][D/32], layers 1..L-1 [MT][H/32], then transposed: layer 0
  // [MT0][H/32], layers 1..L-1 [MT][H/32]
  static constexpr int KX0 = D / 32, KXH = H / 32;
  static constexpr int X_HIDDEN = MT * KX0;
  static constexpr int X_T0 = X_HIDDEN + (L - 1) * MT * KXH;
  static constexpr int X_THIDDEN = X_T0 + MT0 * KXH;
  static constexpr int X_FRAGS = X_THIDDEN + (L - 1) * MT * KXH;
  // the FP16 fragments (the same, then the head's forward ones) end the
  // packed weights, 512 floats each
  static constexpr int64_t F16_BASE = STATS_BASE + 4 * (L + 1);
  static constexpr int F16_FRAGS = X_FRAGS + KXH;
  static constexpr int64_t PACKED = F16_BASE + int64_t(F16_FRAGS) * 512;
};

// out[mt] = relu(W x + b) over the MT m-tiles: fragments A [MT][KT], input x
// in k-tile order, bias b (this layer's H values).
template <int KT, int MT>
__device__ __forceinline__ void dense_relu(const float* __restrict__ A, const float (&x)[KT],
                                           const float* __restrict__ b, float (&y)[4 * MT],
                                           int lane, int g) {
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const f32x4 acc = mfma_chain<KT>(A + mt * KT * 64, x, lane);
    const float4 bb = *reinterpret_cast<const float4*>(b + 16 * mt + 4 * g);
    y[4 * mt + 0] = fmaxf(acc[0] + bb.x, 0.0f);
    y[4 * mt + 1] = fmaxf(acc[1] + bb.y, 0.0f);
    y[4 * mt + 2] = fmaxf(acc[2] + bb.z, 0.0f);
    y[4 * mt + 3] = fmaxf(acc[3] + bb.w, 0.0f);
    tile_fence();
  }
}

// One wave's 16 samples [base, base + 16) through the MLP: x0 (the input in
// k-tile order, zero past M), every hidden layer's output h[l], and the
// head's accumulator z (lanes of group 0 hold the 4 logits of sample c,
// biases not yet added).
template <int D, int H, int L>
__device__ __forceinline__ void forward_tile(const float* __restrict__ emb, int64_t M,
                                             const float* __restrict__ packed, int64_t s,
                                             float (&x0)[D / 4], float (&h)[L][H / 4], f32x4& z,
                                             int lane, int g) {
  using T = TrainDims<D, H, L>;
  const float* bias = packed + T::BIAS_BASE;
#pragma unroll
  for (int t = 0; t < D / 16; ++t) {
    float4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (s < M) v = *reinterpret_cast<const float4*>(emb + s * D + 16 * t + 4 * g);
    x0[4 * t + 0] = v.x;
    x0[4 * t + 1] = v.y;
    x0[4 * t + 2] = v.z;
    x0[4 * t + 3] = v.w;
  }
  dense_relu<T::KT0, T::MT>(packed, x0, bias, h[0], lane, g);
#pragma unroll
  for (int l = 1; l < L; ++l)
    dense_relu<T::KTH, T::MT>(packed + (T::F_HIDDEN + (l - 1) * T::MT * T::KTH) * 64, h[l - 1],
                              bias + l * H, h[l], lane, g);
  z = mfma_chain<T::KTH>(packed + T::F_HEAD * 64, h[L - 1], lane);
}

// ReLU as an integer max on the float's bits (the split-BF16 MLP kernel's).
__device__ __forceinline__ float relu_bits(float x) {
  return __int_as_float(max(__float_as_int(x), 0));
}

// out[s] = (sigma, sigmoid(r), sigmoid(g), sigmoid(b)) of emb[s] for s < M.
// The MLP runs on the FP16 matrix units at FP32 accuracy (F16Mlp); a tile with
// an input that is not finite runs on the FP32 MFMAs (forward_tile, 16 samples
// at a time).  Each block stages the weights in LDS, so a wave takes
// consecutive tiles, the next one's features loaded while it evaluates one.
// Bound: the matrix pipe and the epilogue's vector instructions (mlp_f16x3.h).
// On the FP32 MFMAs, with the fragments from L2, 1,000,003 samples took
// 948 us, now 215; 4,093 samples 42 and 17 us.
template <int D, int H, int L>
__global__ __launch_bounds__(64 * kF16Waves, 1) void mlp_train_forward_kernel(
    const float* __restrict__ emb, int64_t M, const float* __restrict__ packed,
    float* __restrict__ out) {
  using T = TrainDims<D, H, L>;
  constexpr int NT = kF16NT;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const auto mlp = F16Mlp<D, H, L>::stage_packed(packed + T::F16_BASE,
                                                 packed + T::F16_BASE + int64_t(T::X_FRAGS) * 512,
                                                 packed + T::STATS_BASE, packed + T::BIAS_BASE,
                                                 smem_raw);
  const int lane = threadIdx.x & 63, g = lane >> 4, col = lane & 15;
  const int64_t tiles = (M + kF16Samples - 1) / kF16Samples;
  const int64_t waves = int64_t(gridDim.x) * kF16Waves, each = (tiles + waves - 1) / waves;
  const int64_t first = (int64_t(blockIdx.x) * kF16Waves +
                         __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * each;
  const int64_t last = min(first + each, tiles);
  float4 next[NT][D / 16];
  const auto load = [&](int64_t t) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int64_t s = t * kF16Samples + 16 * j + col;
#pragma unroll
      for (int q = 0; q < D / 16; ++q)
        next[j][q] = s < M ? *reinterpret_cast<const float4*>(emb + s * D + 16 * q + 4 * g)
                           : float4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  };
  if (first < last) load(first);
  const bool beyond = mlp.beyond();
  for (int64_t t = first; t < last; ++t) {
    float x[NT][D / 4];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int q = 0; q < D / 16; ++q) {
        x[j][4 * q + 0] = next[j][q].x;
        x[j][4 * q + 1] = next[j][q].y;
        x[j][4 * q + 2] = next[j][q].z;
        x[j][4 * q + 3] = next[j][q].w;
      }
    f32x4 z[NT];
    bool done = false;
    if (!beyond)
      done = mlp.tile(x, lane, g, z, [&](int l) {
        if (l == 1 && t + 1 < last) load(t + 1);
      });
    if (!done) {
      const float4 bb = *reinterpret_cast<const float4*>(packed + T::BIAS_BASE + L * H);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        float x0[T::KT0];
        float h[L][T::KTH];
        forward_tile<D, H, L>(emb, M, opaque(packed), t * kF16Samples + 16 * j + col, x0, h,
                              z[j], lane, g);
        z[j] = z[j] + f32x4{bb.x, bb.y, bb.z, bb.w};
      }
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int64_t s = t * kF16Samples + 16 * j + col;
      if (g == 0 && s < M) {
        float4 o;
        o.x = z[j][0];
        o.y = logistic(z[j][1]);
        o.z = logistic(z[j][2]);
        o.w = logistic(z[j][3]);
        *reinterpret_cast<float4*>(out + s * 4) = o;
      }
    }
  }
}

// Backward: demb [M][D] and this block's partial parameter gradients
// (partial + blockIdx.x * PARAMS, torch order), from dout [M][4] = the
// gradient of (sigma, r, g, b) after the sigmoid.  Needs H == 16 * waves.
// On the FP32 MFMAs, for the chunks of 64 samples that the 16-bit kernel left
// (chunk_flags): returns at once where none of the nflags blocks' flags is set
// (the sum over partials looks at the same flags).
template <int D, int H, int L>
__global__ __launch_bounds__(kTrainBlock) void mlp_train_backward_f32_kernel(
    const float* __restrict__ emb, int64_t M, const float* __restrict__ packed,
    const float* __restrict__ dout, float* __restrict__ demb, float* __restrict__ partial,
    const int32_t* __restrict__ flags, int nflags, const int32_t* __restrict__ chunk_flags) {
  using T = TrainDims<D, H, L>;
  static_assert(T::MT == kTrainWaves, "one hidden m-tile per wave");
  static_assert(D % 16 == 0 && D <= H, "input width");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  float* lds_dz = reinterpret_cast<float*>(smem_raw);    // [128 samples][kLdsRow]
  float* lds_x = lds_dz + kTrainChunk * kLdsRow;          // [128 samples][kLdsRow]
  const int lane = threadIdx.x & 63, g = lane >> 4, col = lane & 15;
  const int w = threadIdx.x >> 6;
  const float* bias = packed + T::BIAS_BASE;
  // this wave's rows of the weight gradients: layer 0 rows 16w.. over the
  // D / 16 input tiles, hidden layers 1..L-1 rows 16w.. over H / 16 tiles,
  // the head's columns 16w..; a bias tile per layer (wave 0: the head's)
  f32x4 gw0[T::MT0], gw[L > 1 ? L - 1 : 1][T::MT], gb[L], gh, ghb;
#pragma unroll
  for (int i = 0; i < T::MT0; ++i) gw0[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int l = 0; l < (L > 1 ? L - 1 : 1); ++l)
#pragma unroll
    for (int i = 0; i < T::MT; ++i) gw[l][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int l = 0; l < L; ++l) gb[l] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  gh = ghb = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  float* my_dz = lds_dz + (w * 16 + col) * kLdsRow;
  float* my_x = lds_x + (w * 16 + col) * kLdsRow;
  int flagged = 0;
  for (int i = threadIdx.x; i < nflags; i += kTrainBlock) flagged |= flags[i];
  if (!__syncthreads_or(flagged)) return;
  const int64_t chunks = (M + kTrainChunk - 1) / kTrainChunk;
  for (int64_t ch = blockIdx.x; ch < chunks; ch += gridDim.x) {
    const int64_t half = ch * kTrainChunk + kBwdChunk;   // the second chunk's first sample
    const bool first = chunk_flags[2 * ch] != 0;
    const bool second = half < M && chunk_flags[2 * ch + 1] != 0;
    if (!first && !second) continue;
    // the samples below `end` are this wave's to do: none of a chunk done before
    const int64_t end = (w < kTrainWaves / 2 ? first : second) ? M : 0;
    const int64_t s = ch * kTrainChunk + w * 16 + col;
    const float* pk = opaque(packed);
    const float* At = pk + T::T_BASE;
    float x0[T::KT0];
    float h[L][T::KTH];
    f32x4 z;
    forward_tile<D, H, L>(emb, end, pk, s, x0, h, z, lane, g);
    // dlogits on the lanes of group 0: d sigma as given, d rgb through the
    // sigmoid's derivative y (1 - y)
    f32x4 dl = {0.0f, 0.0f, 0.0f, 0.0f};
    if (g == 0 && s < end) {
      const float4 d = *reinterpret_cast<const float4*>(dout + s * 4);
      const float4 bb = *reinterpret_cast<const float4*>(bias + L * H);
      const float y1 = logistic(z[1] + bb.y), y2 = logistic(z[2] + bb.z),
                  y3 = logistic(z[3] + bb.w);
      dl[0] = d.x;
      dl[1] = d.y * (y1 * (1.0f - y1));
      dl[2] = d.z * (y2 * (1.0f - y2));
      dl[3] = d.w * (y3 * (1.0f - y3));
    }
    // ---- head: dW_head = dl^T h[L-1], dh = W_head^T dl
    if (g == 0) *reinterpret_cast<f32x4*>(my_dz) = dl;
#pragma unroll
    for (int mt = 0; mt < T::MT; ++mt)
      *reinterpret_cast<f32x4*>(my_x + 16 * mt + 4 * g) = f32x4{
          h[L - 1][4 * mt], h[L - 1][4 * mt + 1], h[L - 1][4 * mt + 2], h[L - 1][4 * mt + 3]};
    __syncthreads();
#pragma unroll 1
    for (int kk = 0; kk < kTrainChunk / 4; ++kk) {
      const int row = (4 * kk + g) * kLdsRow;
      const float a = col < 4 ? lds_dz[row + col] : 0.0f;
      gh = mfma4(a, lds_x[row + 16 * w + col], gh);
      if (w == 0) ghb = mfma4(a, 1.0f, ghb);
    }
    __syncthreads();
    float dh[T::KTH];
    {
      // operand B of W_head^T: lane group g takes logit g of sample c
      const float t0 = __shfl(dl[0], col, 64), t1 = __shfl(dl[1], col, 64),
                  t2 = __shfl(dl[2], col, 64), t3 = __shfl(dl[3], col, 64);
      const float b = g == 0 ? t0 : (g == 1 ? t1 : (g == 2 ? t2 : t3));
#pragma unroll
      for (int mt = 0; mt < T::MT; ++mt) {
        const f32x4 acc =
            mfma4(At[(T::T_HEAD + mt) * 64 + lane], b, f32x4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
        for (int r = 0; r < 4; ++r) dh[4 * mt + r] = acc[r];
        tile_fence();
      }
    }
    // ---- hidden layers, last to first: layer l maps h[l-1] (x0 for l = 0)
    // to h[l]
#pragma unroll
    for (int l = L - 1; l >= 0; --l) {
      float dz[T::KTH];
#pragma unroll
      for (int k = 0; k < T::KTH; ++k) dz[k] = h[l][k] > 0.0f ? dh[k] : 0.0f;
#pragma unroll
      for (int mt = 0; mt < T::MT; ++mt)
        *reinterpret_cast<f32x4*>(my_dz + 16 * mt + 4 * g) =
            f32x4{dz[4 * mt], dz[4 * mt + 1], dz[4 * mt + 2], dz[4 * mt + 3]};
      if (l > 0) {
        // the first layer's output again, from x0: keeping it from the
        // forward pass would hold 32 more registers through every later phase
        if (l == 1) dense_relu<T::KT0, T::MT>(opaque(packed), x0, bias, h[0], lane, g);
#pragma unroll
        for (int mt = 0; mt < T::MT; ++mt)
          *reinterpret_cast<f32x4*>(my_x + 16 * mt + 4 * g) =
              f32x4{h[l - 1][4 * mt], h[l - 1][4 * mt + 1], h[l - 1][4 * mt + 2],
                    h[l - 1][4 * mt + 3]};
      } else {
#pragma unroll
        for (int t = 0; t < T::MT0; ++t)
          *reinterpret_cast<f32x4*>(my_x + 16 * t + 4 * g) =
              f32x4{x0[4 * t], x0[4 * t + 1], x0[4 * t + 2], x0[4 * t + 3]};
      }
      __syncthreads();
      // weight gradient rows 16w..16w+15 of layer l, 4 samples per step
#pragma unroll 1
      for (int kk = 0; kk < kTrainChunk / 4; ++kk) {
        const int row = (4 * kk + g) * kLdsRow;
        const float a = lds_dz[row + 16 * w + col];
        if (l > 0) {
#pragma unroll
          for (int mi = 0; mi < T::MT; ++mi)
            gw[l > 0 ? l - 1 : 0][mi] = mfma4(a, lds_x[row + 16 * mi + col],
                                              gw[l > 0 ? l - 1 : 0][mi]);
        } else {
#pragma unroll
          for (int mi = 0; mi < T::MT0; ++mi)
            gw0[mi] = mfma4(a, lds_x[row + 16 * mi + col], gw0[mi]);
        }
        gb[l] = mfma4(a, 1.0f, gb[l]);
      }
      __syncthreads();
      if (l > 0) {
        const float* A = At + (T::T_HIDDEN + (l - 1) * T::MT * T::KTH) * 64;
#pragma unroll
        for (int mt = 0; mt < T::MT; ++mt) {
          const f32x4 acc = mfma_chain<T::KTH>(A + mt * T::KTH * 64, dz, lane);
#pragma unroll
          for (int r = 0; r < 4; ++r) dh[4 * mt + r] = acc[r];
          tile_fence();
        }
      } else {
#pragma unroll
        for (int mt = 0; mt < T::MT0; ++mt) {
          const f32x4 acc = mfma_chain<T::KTH>(At + mt * T::KTH * 64, dz, lane);
          if (s < end) *reinterpret_cast<f32x4*>(demb + s * D + 16 * mt + 4 * g) = acc;
          tile_fence();
        }
      }
    }
  }
  // this block's partial sums, in torch order
  float* P = partial + int64_t(blockIdx.x) * T::PARAMS;
  const int o = 16 * w + 4 * g;  // hidden output rows o..o+3 of this lane
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int mi = 0; mi < T::MT0; ++mi) P[T::P_W0 + int64_t(o + r) * D + 16 * mi + col] = gw0[mi][r];
    if (col == 0) P[T::P_B0 + o + r] = gb[0][r];
#pragma unroll
    for (int l = 1; l < L; ++l) {
      const int64_t base = T::P_LAYER1 + int64_t(l - 1) * (int64_t(H) * H + H);
#pragma unroll
      for (int mi = 0; mi < T::MT; ++mi) P[base + int64_t(o + r) * H + 16 * mi + col] = gw[l - 1][mi][r];
      if (col == 0) P[base + int64_t(H) * H + o + r] = gb[l][r];
    }
    if (g == 0) {
      P[T::P_HEAD + int64_t(r) * H + 16 * w + col] = gh[r];
      if (w == 0 && col == 0) P[T::P_HEAD + 4 * H + r] = ghb[r];
    }
  }
}

// ---------------------------------------------------------------------------
// The backward kernel on the 16-bit matrix units: FP16 hi / lo parts (FP32
// accuracy, as in mlp_f16x3.h) or, for FieldMLPx3, split BF16.
//
// A block of 8 waves takes 64 samples at a time.  The layers' outputs live in
// LDS as hi and lo planes of [feature][sample]; wave w computes output
// features 16w..16w+15 of every layer for all 64 samples, so a layer's
// weights are read once per block and 64 samples (each wave its own 8 KB from
// L2, loaded while the previous layer ends) where a wave per 16 samples read
// all 288 KB for each of them.  A layer's products run as Y = X W^T, so a
// lane's accumulator holds four consecutive samples of one feature and goes
// out as one 8-byte store per part; the next layer's operand (8 features of a
// sample) comes back through the transposing LDS read (ds_read_b64_tr_b16),
// and the weight gradients' operands (8 samples of a feature) are plain
// 16-byte reads of the same planes.  Rows are padded to 72 halves (36 banks);
// unpadded rows with their units permuted by row gave the same conflicts and
// needed an address register per tile.
//
//   phases (a barrier after each): the chunk's features; layers 0, 1, 2; the
//   head with the logits' gradients; dz2 (dW_head); dW_2 and dz1; dW_1 and
//   dz0; dW_0 and the input gradient.
//
// dz2 takes the plane set of no layer, dz1 takes h2's and dz0 takes dz2's,
// which are dead by then.  The ReLU masks stay in registers (a bit per value).
// The weight gradients accumulate in registers over the whole kernel, a wave
// holding 32 x 64 of each hidden layer's, 16 x 32 of the first's and 4 x 16 of
// the head's; the bias gradients are FP32 sums of dz, and the head's weight
// gradient (FP16 form) FP32 sums of the vector unit.  Block partials are
// added in block order, so the gradients do not depend on timing.
//
// Scales (FP16 only; all powers of two, exact).  Weights as in mlp_f16x3.h.  A
// sample's activations are scaled by a bound of its layer's outputs, from the
// layers' largest row sums |W| and biases: one layer past the sample's
// largest feature for h0, two for h1, and for h2 two past its largest h0 (an
// FP16 pair covers 2^40, so a loose bound costs no accuracy until it is 2^17
// too large).  The logits' gradients of a sample are divided by the power of
// two below their largest, everything behind them is linear in it, and the
// bounds of dz are then the same for every sample; the input gradient is
// multiplied back.  In the weight gradients, sums over samples, each sample's
// factor multiplies dz when it is read, in bands of samples of like size
// (BwdBands).
// The matrix unit's long sums come out low on average (measured: every bias
// gradient's error negative, whatever its own sign; one accumulation by itself
// rounds to nearest).  That is below FP32's rounding in one product, but a
// parameter's gradient adds a million: so a chunk's sums are added by the
// vector unit, and every second sample's normalised gradient, and every second
// chunk's weight gradient, is computed with the other sign.  (In one accumulator
// the weight gradients were 4e-6 off on a million samples, with one sign the
// bias gradients 3e-6, FP32 MFMAs 1e-6.)
// A chunk with an operand that is not finite or outside 2^-40 .. 2^60 is found
// out before its weight gradients and left to the FP32 kernel above, which adds
// partial sums of its own (all chunks, if it is a weight).  Repeating the whole
// call there, a million samples with one such sample took 4,376 us where all on
// the FP32 MFMAs had taken 3,975.
//
// Bound: LDS reads (about 15 k cycles per 64 samples at 128 B per cycle)
// beside 12.5 k of MFMAs, and the phases' barriers.
// Against the form before (each wave its own 16 samples, all weights from L2 for
// each): FP32 2,970 -> 1,367 us per million samples whose gradients spread over
// four decades, 4,093 samples 109 -> 36 us; split BF16 686 -> 475 us for the
// 0.51 M samples of a training step of 8,192 rays.  The FP32 gradients are
// 6.3e-7 off 64 bits at most (a million samples, eight networks), 3.0e-6 before.
constexpr int kBwdWaves = 8;
constexpr int kBwdBlock = 64 * kBwdWaves;
constexpr int kBwdRow = 72;                  // halves per plane row
constexpr int kBwdPlane = 128 * kBwdRow;     // halves per hidden plane
constexpr int kBwdPlane0 = 32 * kBwdRow;     // halves per input plane

typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(4))) short s16x4;

struct BwdLds {
  unsigned short x0[2 * kBwdPlane0];         // input: hi plane, lo plane
  unsigned short t[4][2 * kBwdPlane];        // h0, h1, h2, dz2 (split BF16: h2 in FP32 before)
  float dl[kBwdChunk][4];                    // logits' gradients (normalised)
  union {
    unsigned short head[2][4][4][4][8];      // head weights hi / lo: [kt][g][logit][i]
    float head32[32][4][4];                  // split BF16: FP32, [k-tile of 4][g][logit]
  };
  float back[4][kBwdChunk];                  // accumulator -> sum, layers 0..2 and head
  float scale[3][kBwdChunk];                 // sum -> parts, h0, h1, h2
  _Float16 factor[kBwdWaves][kBwdChunk];     // each wave's sample factors of a weight gradient
  float unit[kBwdChunk];                     // 2^k of the normalised gradients (0: none)
  int top0[kBwdChunk];                       // largest h0 (float bits)
  short dz_top[3][kBwdWaves][4];             // largest |dz| of each wave's lane groups (upper 16 bits)
  int wild;
};
static_assert(sizeof(BwdLds) <= 160 * 1024, "LDS");

template <bool F16>
__device__ __forceinline__ f32x4 mm16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// a * b as split parts, hi b_lo, lo b_hi, hi b_hi (for BF16 the forward
// kernel's order: Wl Xh, Wh Xl, Wh Xh with W in b).
template <bool F16>
__device__ __forceinline__ f32x4 mm16x3(u32x4 ah, u32x4 al, u32x4 bh, u32x4 bl, f32x4 c) {
  c = mm16<F16>(ah, bl, c);
  c = mm16<F16>(al, bh, c);
  return mm16<F16>(ah, bh, c);
}

// Parts of s0 a and s1 b as packed pairs (BF16: s0 = s1 = 1).
template <bool F16>
__device__ __forceinline__ void parts2(float a, float b, float s0, float s1, unsigned int& hi,
                                       unsigned int& lo) {
  if constexpr (F16) {
    f16x2 h, l;
    f16_split2(a, b, s0, s1, h, l);
    hi = __builtin_bit_cast(unsigned int, h);
    lo = __builtin_bit_cast(unsigned int, l);
  } else {
    split2(a, b, hi, lo);
  }
}

__device__ __forceinline__ u32x4 lds128(const unsigned short* p) {
  return *reinterpret_cast<const u32x4*>(p);
}

// Halves from a plane's start to (row r, sample i).
__device__ __forceinline__ int bwd_at(int r, int i) { return r * kBwdRow + i; }

// An operand of 8 features of a lane's sample, transposed out of a plane of
// [feature][sample] rows: p = the lane's address (row 4 g + i / 4, sample
// 4 (i % 4), i = lane % 16) of the k-tile's first half; the second is 16 rows
// on.  Lane (g, c) gets features 4 g + 0..3 and 16 + 4 g + 0..3 of sample c.
__device__ __forceinline__ u32x4 lds_tr(const unsigned short* p) {
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 16 * kBwdRow));
  const u32x2 x = __builtin_bit_cast(u32x2, a), y = __builtin_bit_cast(u32x2, b);
  return u32x4{x[0], x[1], y[0], y[1]};
}

typedef const __attribute__((address_space(1))) u32x4* global_u32x4;

// The wave's weight fragments of a layer: KT pairs at F (fragment: 64 lanes of
// hi, then of lo).
template <int KT>
struct BwdFrags {
  u32x4 h[KT], l[KT];
  __device__ __forceinline__ void load(global_u32x4 F, int lane) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      h[kt] = F[128 * kt + lane];
      l[kt] = F[128 * kt + 64 + lane];
    }
  }
};

// acc[m] += the layer's products for samples 16 m.. over KT k-tiles: operand
// planes at p + at[m] (the lane's transposing address; lo plane `lo` halves on).  The
// four sample tiles' chains alternate; a scheduling barrier closes each k-tile
// (the SIMD's other wave covers its reads: a second set of operands in
// registers was spilled).  FP16: the small products have sums of their own, so
// that only KT accumulations round at the result's size.
template <bool F16, int KT>
__device__ __forceinline__ void bwd_layer(const unsigned short* p, const int (&at)[4], int lo,
                                          const BwdFrags<KT>& w, f32x4 (&acc)[4]) {
  f32x4 small[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) small[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) {
    u32x4 ah[4], al[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) ah[m] = lds_tr(p + at[m] + kt * 32 * kBwdRow);
#pragma unroll
    for (int m = 0; m < 4; ++m) al[m] = lds_tr(p + at[m] + kt * 32 * kBwdRow + lo);
#pragma unroll
    for (int m = 0; m < 4; ++m)
      (F16 ? small[m] : acc[m]) = mm16<F16>(ah[m], w.l[kt], F16 ? small[m] : acc[m]);
#pragma unroll
    for (int m = 0; m < 4; ++m)
      (F16 ? small[m] : acc[m]) = mm16<F16>(al[m], w.h[kt], F16 ? small[m] : acc[m]);
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[m] = mm16<F16>(ah[m], w.h[kt], acc[m]);
    tile_fence();
  }
  if constexpr (F16) {
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[m] = acc[m] + small[m];
  }
}

// The samples of a chunk in bands of like size, for a sum over samples whose
// terms are 2^q[lane] x operands of one scale: each step takes those within
// 2^-kBand of the largest that are left, leaves their factors +-2^(q - top) in
// the wave's row of LDS (0 for the others) and top in `top`; false when none
// are left.  u: the samples' units (0: no gradient), us: their signs.
// A factor multiplies the FP16 parts of an operand, whose low parts lose bits
// to FP16's subnormals where it is small; in one band for the whole chunk, a
// sample 2^-25 of the largest would vanish, also from the rows of a weight
// gradient that the larger samples do not reach.  Gradients fall along a ray
// with its transmittance, so samples that far apart are common.
// Rows of dW that only samples 2^-k of their neighbours' reach, error against
// 64 bits (root mean square over 12 networks): up to 5.5e-7 for every k with 16,
// where the FP32 MFMAs' is 6.4e-7; with 18, 3.3e-6 at k = 17, with 20, 1.1e-5 at
// k = 19, with one band all of the row from k = 25 on.  A million samples whose
// gradients spread over four decades, forward and backward: 1,467 us with 16,
// 1,377 with 18, 1,366 with 20.
constexpr int kBand = 16;
struct BwdBands {
  int q;
  float us;
  bool left;
  int top;
  __device__ __forceinline__ BwdBands(int q_, float u, float sign)
      : q(q_), us(copysignf(sign, u * sign)), left(u != 0.0f), top(0) {}
  __device__ __forceinline__ bool next(_Float16* factor, int lane) {
    if (!__any(left)) return false;
    top = wave_max(left ? q : 0);   // exponents are positive
    const int d = q - top;
    const bool in = left && d > -kBand;
    wave_sync();   // the band before has been read
    factor[lane] = in ? _Float16(us * __int_as_float((127 + d) << 23)) : _Float16(0.0f);
    wave_sync();
    left = left && !in;
    return true;
  }
};

// sum[a][b] += 2^e x the sum over a band's samples of rows A (dz, NA tiles
// of 16) and B (the layer's input, NB tiles): rows from pa / pb on, the lane's
// at[ks] halves on (row c, sample 32 ks + 8 g), lo planes `lo_a` / `lo_b` halves
// on; factor: the samples' factors, multiplied by 2^up (what the rows leave of
// FP16's range: the bound that dz was scaled by is loose, by some 2^10 for dz0);
// by: their sign in this chunk.
template <bool F16, int NA, int NB>
__device__ __forceinline__ void bwd_dw(const unsigned short* pa, int lo_a,
                                       const unsigned short* pb, int lo_b, const int (&at)[2],
                                       const _Float16* factor, int up, int g, int e, float by,
                                       f32x4 (&sum)[NA][NB]) {
  constexpr int KS = kBwdChunk / 32;
  u32x4 ah[KS][NA], al[KS][NA];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      ah[ks][a] = lds128(pa + at[ks] + a * 16 * kBwdRow);
      al[ks][a] = lds128(pa + at[ks] + a * 16 * kBwdRow + lo_a);
    }
  if constexpr (F16) {
    const _Float16 raise = _Float16(__int_as_float((127 + up) << 23));
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const f16x8 f = *reinterpret_cast<const f16x8*>(factor + 32 * ks + 8 * g) * raise;
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        ah[ks][a] = __builtin_bit_cast(u32x4, __builtin_bit_cast(f16x8, ah[ks][a]) * f);
        al[ks][a] = __builtin_bit_cast(u32x4, __builtin_bit_cast(f16x8, al[ks][a]) * f);
      }
    }
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    f32x4 acc[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const u32x4 bh = lds128(pb + at[ks] + b * 16 * kBwdRow);
      const u32x4 bl = lds128(pb + at[ks] + b * 16 * kBwdRow + lo_b);
#pragma unroll
      for (int a = 0; a < NA; ++a) acc[a] = mm16<F16>(ah[ks][a], bl, acc[a]);
#pragma unroll
      for (int a = 0; a < NA; ++a) acc[a] = mm16<F16>(al[ks][a], bh, acc[a]);
#pragma unroll
      for (int a = 0; a < NA; ++a) acc[a] = mm16<F16>(ah[ks][a], bh, acc[a]);
    }
    tile_fence();
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sum[a][b][r] = F16 ? __fmaf_rn(__builtin_amdgcn_ldexpf(acc[a][r], e), by, sum[a][b][r])
                           : sum[a][b][r] + acc[a][r];
    // the sums as values of this place: the compiler would otherwise move the
    // additions to the end of the step and keep both operands until then
#pragma unroll
    for (int a = 0; a < NA; ++a) asm volatile("" : "+v"(sum[a][b]));
  }
}

// Exponent window of the FP16 form's operands, 2^-40 to 2^60 (or 0): every
// factor formed from two of them is a normal number.
constexpr int kTameLow = 87, kTameHigh = 187;
__device__ __forceinline__ bool tame(float v) {
  const int e = int(__float_as_uint(v) >> 23);
  return v == 0.0f || (e >= kTameLow && e <= kTameHigh);
}
__device__ __forceinline__ int tame_exponent(float v) {
  return min(max(int(__float_as_uint(v) >> 23), kTameLow), kTameHigh);
}
// The exponent e of f16_unscale(e) * f16_unscale(ew).
__device__ __forceinline__ int feature_exponent(float back, int ew) {
  return (__float_as_int(back) >> 23) + 127 - (ew - 14) + 14;
}

template <int D, int H, int L, bool F16>
__global__ __launch_bounds__(kBwdBlock, 1) void mlp_train_backward_kernel(
    const float* __restrict__ emb, int64_t M, const float* __restrict__ packed,
    const u32x4* __restrict__ frags, const float* __restrict__ dout, float* __restrict__ demb,
    float* __restrict__ partial, int32_t* __restrict__ flags,
    int32_t* __restrict__ chunk_flags) {
  using T = TrainDims<D, H, L>;
  static_assert(D == 32 && H == 128 && L == 3, "the phases below");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  BwdLds& S = *reinterpret_cast<BwdLds*>(smem_raw);
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const float* bias = packed + T::BIAS_BASE;

  // the layers' weight exponents and bounds (FP16)
  [[maybe_unused]] int ew[4] = {0, 0, 0, 0};
  [[maybe_unused]] float rowsum[4], maxb[4];
  [[maybe_unused]] int ez[3] = {0, 0, 0};   // exponents of dz2, dz1, dz0
  bool wild_weights = false;
  if constexpr (F16) {
    const float* st = packed + T::STATS_BASE;
    float bound = 2.0f;   // of the normalised logits' gradients
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      wild_weights = wild_weights || !tame(st[l]) || !tame(st[4 + l]) || !tame(st[8 + l]) ||
             !(st[12 + l] <= 0x1p60f);
      ew[l] = tame_exponent(st[l]);
      rowsum[l] = st[4 + l];
      maxb[l] = st[12 + l];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {   // dz2 through the head, dz1 through W_2, dz0 through W_1
      bound = bound * st[8 + 3 - k];
      wild_weights = wild_weights || !tame(bound);
      ez[k] = tame_exponent(bound);
    }
  }
  // the head's weights in LDS (operand of the logits; packed head fragment mt,
  // lane (o, c) = W[o][16 mt + c])
  const float* WT = packed + T::T_BASE + T::T_HEAD * 64;
  const auto head_weight = [WT](int o, int f) { return WT[(f >> 4) * 64 + o * 16 + (f & 15)]; };
  for (int i = threadIdx.x; F16 && i < 4 * 4 * 4 * 4; i += kBwdBlock) {
    // pair p of logit o, k-tile kt, group gg: features 32 kt + {4 gg + ..}
    const int p = i & 3, o = (i >> 2) & 3, gg = (i >> 4) & 3, kt = i >> 6;
    const int j = 2 * p, f = 32 * kt + (j < 4 ? 4 * gg + j : 16 + 4 * gg + j - 4);
    const float s = f16_scale(ew[3]);
    unsigned int hi, lo;
    parts2<F16>(head_weight(o, f), head_weight(o, f + 1), s, s, hi, lo);
    *reinterpret_cast<unsigned int*>(&S.head[0][kt][gg][o][j]) = hi;
    *reinterpret_cast<unsigned int*>(&S.head[1][kt][gg][o][j]) = lo;
  }
  for (int i = threadIdx.x; !F16 && i < 32 * 4 * 4; i += kBwdBlock)
    // k-tile kt = 4 t + r: feature 16 t + 4 g + r
    S.head32[i >> 4][(i >> 2) & 3][i & 3] =
        head_weight(i & 3, 16 * (i >> 6) + 4 * ((i >> 2) & 3) + ((i >> 4) & 3));
  // this lane's biases (feature c of the wave's, logit c of the head) and head
  // weights
  float bl[3], bh;
#pragma unroll
  for (int l = 0; l < 3; ++l) bl[l] = bias[l * H + 16 * w + c];
  bh = bias[L * H + (c & 3)];
  float wh[4];
#pragma unroll
  for (int o = 0; o < 4; ++o)
    wh[o] = packed[T::T_BASE + (T::T_HEAD + w) * 64 + o * 16 + c];
  bool flagged = F16 && wild_weights;   // a chunk was left to the FP32 kernel
  for (int i = threadIdx.x; i < kBwdChunk; i += kBwdBlock) S.top0[i] = 0;

  const f32x4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 gw2[2][4], gw1[2][4], gw0[1][2], gh = zero4;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) gw2[a][b] = gw1[a][b] = zero4;
  gw0[0][0] = gw0[0][1] = zero4;
  float gb[3] = {0.0f, 0.0f, 0.0f}, ghb = 0.0f;

  const int64_t chunks = (M + kBwdChunk - 1) / kBwdChunk;
  // the chunk's features: thread (sample, features 4 j..) = threadIdx / 8, % 8
  const int xs = threadIdx.x >> 3, xj = threadIdx.x & 7;
  float4 xin = {0.0f, 0.0f, 0.0f, 0.0f};
  const auto load_x = [&](int64_t ch) {
    const int64_t s = ch * kBwdChunk + xs;
    xin = (ch < chunks && s < M) ? *reinterpret_cast<const float4*>(emb + s * D + 4 * xj)
                                 : float4{0.0f, 0.0f, 0.0f, 0.0f};
  };
  load_x(blockIdx.x);
  __syncthreads();

  // weights beyond the window leave every chunk
  for (int64_t ch = blockIdx.x + int64_t(threadIdx.x) * gridDim.x; flagged && ch < chunks;
       ch += int64_t(gridDim.x) * kBwdBlock)
    chunk_flags[ch] = 1;
  for (int64_t ch = flagged ? chunks : blockIdx.x; ch < chunks; ch += gridDim.x) {
    [[maybe_unused]] bool wild = false;
    const int64_t s0 = ch * kBwdChunk;
    const float sign = (ch / gridDim.x) & 1 ? -1.0f : 1.0f;   // of the chunk's weight gradients
    // the lane index as a value of this step: the addresses formed from it
    // would otherwise be kept from step to step, and spilled
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const int g = lane >> 4, c = lane & 15;
    // lane addresses in a plane: transposing (layers, per sample tile), own
    // store (feature row 16 w + c, samples 4 g of each tile), rows of the weight
    // gradients (row c, samples 8 g of each half)
    int at_tr[4], at_out[4], at_row[2];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      at_tr[m] = bwd_at(4 * g + (c >> 2), 16 * m + 4 * (c & 3));
      at_out[m] = 16 * w * kBwdRow + bwd_at(c, 16 * m + 4 * g);
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) at_row[ks] = bwd_at(c, 32 * ks + 8 * g);
    // global memory for certain: behind opaque() the address would be generic,
    // and a generic load also waits for the LDS
    const global_u32x4 F = (global_u32x4)opaque(frags);
    // ---- the features' parts and the sample's scales
    {
      float sx = 1.0f;
      if constexpr (F16) {
        int m = 0;
        m = max(m, __float_as_int(xin.x) & 0x7FFFFFFF);
        m = max(m, __float_as_int(xin.y) & 0x7FFFFFFF);
        m = max(m, __float_as_int(xin.z) & 0x7FFFFFFF);
        m = max(m, __float_as_int(xin.w) & 0x7FFFFFFF);
        m = max(m, __builtin_amdgcn_mov_dpp(m, 0xB1, 0xF, 0xF, true));
        m = max(m, __builtin_amdgcn_mov_dpp(m, 0x4E, 0xF, 0xF, true));
        m = max(m, __builtin_amdgcn_mov_dpp(m, 0x141, 0xF, 0xF, true));
        const float xm = __int_as_float(m);
        wild = wild || !tame(xm);
        const int ex = tame_exponent(xm);
        sx = f16_scale(ex);
        const float t0 = __fmaf_rn(rowsum[0], xm, maxb[0]) * 1.001f;
        const float t1 = __fmaf_rn(rowsum[1], t0, maxb[1]) * 1.001f;
        wild = wild || !(t0 <= 0x1p60f) || !(t1 <= 0x1p60f);
        const int e0 = tame_exponent(t0), e1 = tame_exponent(t1);
        if (xj == 0) {
          S.back[0][xs] = f16_unscale(ex) * f16_unscale(ew[0]);
          S.scale[0][xs] = f16_scale(e0);
          S.back[1][xs] = f16_unscale(e0) * f16_unscale(ew[1]);
          S.scale[1][xs] = f16_scale(e1);
          S.back[2][xs] = f16_unscale(e1) * f16_unscale(ew[2]);
        }
      }
      unsigned int h0, l0, h1, l1;
      parts2<F16>(xin.x, xin.y, sx, sx, h0, l0);
      parts2<F16>(xin.z, xin.w, sx, sx, h1, l1);
      const unsigned int hv[2] = {h0, h1}, lv[2] = {l0, l1};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        unsigned short* q = &S.x0[bwd_at(4 * xj + k, xs)];
        q[0] = static_cast<unsigned short>(hv[k >> 1] >> 16 * (k & 1));
        q[kBwdPlane0] = static_cast<unsigned short>(lv[k >> 1] >> 16 * (k & 1));
      }
    }
    BwdFrags<1> f0;
    f0.load(F + 128 * w, lane);
    load_x(ch + gridDim.x);
    // the outputs' gradients that waves 0-3 need at the head
    float dy[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (w < 4) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t s = s0 + 16 * w + 4 * g + r;
        if (s < M) dy[r] = dout[s * 4 + (c & 3)];
      }
    }
    BwdFrags<4> f;
    __syncthreads();
    if (threadIdx.x == 0) S.wild = 0;   // read by all before, set at the head

    // relu(z) of an accumulator into plane set l, the mask bits, and (F16) the
    // samples' largest value for layer 0
    unsigned int mask[3];
    const auto forward_out = [&](f32x4 (&acc)[4], int l) {
      unsigned int bits = 0;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        f32x4 sc = {1.0f, 1.0f, 1.0f, 1.0f};
        float h[4];
        if constexpr (F16) {
          const f32x4 bk = *reinterpret_cast<const f32x4*>(&S.back[l][16 * m + 4 * g]);
          sc = *reinterpret_cast<const f32x4*>(&S.scale[l][16 * m + 4 * g]);
#pragma unroll
          for (int r = 0; r < 4; ++r) h[r] = fmaxf(__fmaf_rn(acc[m][r], bk[r], bl[l]), 0.0f);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) h[r] = relu_bits(acc[m][r]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) bits |= (h[r] > 0.0f ? 1u : 0u) << (4 * m + r);
        u32x2 hi, lo;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          unsigned int hw, lw;
          parts2<F16>(h[2 * p], h[2 * p + 1], sc[2 * p], sc[2 * p + 1], hw, lw);
          hi[p] = hw;
          lo[p] = lw;
        }
        *reinterpret_cast<u32x2*>(&S.t[l][at_out[m]]) = hi;
        *reinterpret_cast<u32x2*>(&S.t[l][kBwdPlane + at_out[m]]) = lo;
        if (!F16 && l == 2)
          *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(S.t[3]) + at_out[m]) =
              f32x4{h[0], h[1], h[2], h[3]};
        if constexpr (F16) {
          if (l == 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int top = row_max15(__float_as_int(h[r]));
              if (c == 15) atomicMax(&S.top0[16 * m + 4 * g + r], top);
            }
          }
        }
        tile_fence();
      }
      mask[l] = bits;
    };
    const auto start = [&](f32x4 (&acc)[4], int l) {
      // BF16: the bias is the initial accumulator, as in the forward kernel
      const float b = F16 ? 0.0f : bl[l];
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[m] = f32x4{b, b, b, b};
    };

    // ---- layers 0, 1, 2
    f32x4 acc[4];
    start(acc, 0);
    bwd_layer<F16, 1>(S.x0, at_tr, kBwdPlane0, f0, acc);
    f.load(F + 128 * (T::X_HIDDEN + w * T::KXH), lane);
    forward_out(acc, 0);
    __syncthreads();
    if constexpr (F16) {
      // h2's scale, two layers past the sample's largest h0
      if (threadIdx.x < kBwdChunk) {
        const float t1 = __fmaf_rn(rowsum[1], __int_as_float(S.top0[threadIdx.x]), maxb[1]);
        const float t2 = __fmaf_rn(rowsum[2], t1 * 1.001f, maxb[2]) * 1.001f;
        wild = wild || !(t2 <= 0x1p60f);
        const int e2 = tame_exponent(t2);
        S.scale[2][threadIdx.x] = f16_scale(e2);
        S.back[3][threadIdx.x] = f16_unscale(e2) * f16_unscale(ew[3]);
      }
    }
    start(acc, 1);
    bwd_layer<F16, 4>(S.t[0], at_tr, kBwdPlane, f, acc);
    f.load(F + 128 * (T::X_HIDDEN + (T::MT + w) * T::KXH), lane);
    forward_out(acc, 1);
    __syncthreads();
    start(acc, 2);
    bwd_layer<F16, 4>(S.t[1], at_tr, kBwdPlane, f, acc);
    // W_2^T for dz1
    f.load(F + 128 * (T::X_THIDDEN + (T::MT + w) * T::KXH), lane);
    forward_out(acc, 2);
    __syncthreads();

    // ---- the head: wave m takes samples 16 m..; lanes c < 4 hold logit c of
    // samples 4 g + r
    [[maybe_unused]] float hb = 0.0f;   // of the chunk
    if (w < 4) {
      f32x4 z = zero4;
      if constexpr (F16) {
        const int at_w = bwd_at(4 * g + (c >> 2), 16 * w + 4 * (c & 3));
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
          const unsigned short* p = &S.t[2][at_w + kt * 32 * kBwdRow];
          const u32x4 ah = lds_tr(p), al = lds_tr(p + kBwdPlane);
          const u32x4 bh = lds128(S.head[0][kt][g][c & 3]), bl = lds128(S.head[1][kt][g][c & 3]);
          z = mm16x3<F16>(ah, al, bh, bl, z);
        }
        const f32x4 bk = *reinterpret_cast<const f32x4*>(&S.back[3][16 * w + 4 * g]);
#pragma unroll
        for (int r = 0; r < 4; ++r) z[r] = __fmaf_rn(z[r], bk[r], bh);
      } else {
        // in FP32: logits from parts of h2 and the weights put 2-10% on the
        // error of every gradient against 64 bits (FP32 costs 45 us more per
        // million samples, of 1,150 forward and backward; as FMAs of the vector
        // unit, a lane a quarter of a sample's features, 54)
        const float* h2 = reinterpret_cast<const float*>(S.t[3]);
#pragma unroll
        for (int kt = 0; kt < 32; ++kt) {
          z = mfma4(h2[bwd_at(16 * (kt >> 2) + 4 * g + (kt & 3), 16 * w + c)],
                    S.head32[kt][g][c & 3], z);
          if (kt % 8 == 7) tile_fence();
        }
        z = z + f32x4{bh, bh, bh, bh};
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * w + 4 * g + r;
        const float d = dy[r];
        const float y = logistic(z[r]);
        float v = (c & 3) == 0 ? d : d * (y * (1.0f - y));
        if (c < 4) (F16 ? hb : ghb) += v;
        if constexpr (F16) {
          int m = __float_as_int(v) & 0x7FFFFFFF;
          m = max(m, __builtin_amdgcn_mov_dpp(m, 0xB1, 0xF, 0xF, true));
          m = max(m, __builtin_amdgcn_mov_dpp(m, 0x4E, 0xF, 0xF, true));
          const int e = max(m >> 23, 1);
          wild = wild || e > kTameHigh;
          // 2^(127 - e) and back, negative for odd samples
          const int odd = int(uint32_t(r & 1) << 31);
          v = v * __int_as_float(((254 - min(e, 253)) << 23) | odd);
          if (c == 0) S.unit[i] = m == 0 ? 0.0f : __int_as_float((min(e, 253) << 23) | odd);
        }
        if (c < 4) S.dl[i][c] = v;
      }
    }
    if constexpr (F16) {
      if (wild) S.wild = 1;
    }
    __syncthreads();
    if constexpr (F16) {
      // the chunk to the FP32 kernel; nothing of it is in the sums yet
      const bool skip = __builtin_amdgcn_readfirstlane(S.wild) != 0;
      if (threadIdx.x == 0) chunk_flags[ch] = skip;
      if (skip) {
        flagged = true;
        if (threadIdx.x < kBwdChunk) S.top0[threadIdx.x] = 0;
        continue;
      }
      ghb += hb;
    }

    // the samples' exponents in layer k's weight gradient: those of the
    // normalised gradient times the layer's input
    const auto bands = [&](int k) {
      const float u = S.unit[lane];
      const int e = (__float_as_int(u) & 0x7FFFFFFF) >> 23;
      return BwdBands(e + (k == 0 ? feature_exponent(S.back[0][lane], ew[0])
                                  : 268 - (__float_as_int(S.scale[k > 0 ? k - 1 : 0][lane]) >> 23)),
                      u, sign);
    };
    const auto weight_gradient = [&](auto layer, const unsigned short* pa,
                                     const unsigned short* pb, int lo_b, auto& sum) {
      constexpr int k = layer();
      constexpr int NA = std::extent<std::remove_reference_t<decltype(sum)>, 0>::value;
      constexpr int NB = std::extent<std::remove_reference_t<decltype(sum)>, 1>::value;
      if constexpr (F16) {
        BwdBands b = bands(k);
        // the rows' headroom: those of two waves, or (dz0) of this one
        const short* t = k == 0 ? S.dz_top[0][w] : S.dz_top[k][2 * (w & 3)];
        int top = 0;
#pragma unroll
        for (int i = 0; i < (k == 0 ? 4 : 8); ++i) top = max(top, int(t[i]));
        const int up = min(max(ez[2 - k] - (__builtin_amdgcn_readfirstlane(top) >> 7), 0), 15);
        while (b.next(S.factor[w], lane))
          bwd_dw<true, NA, NB>(pa, kBwdPlane, pb, lo_b, at_row, S.factor[w], up, g,
                               b.top + ez[2 - k] - 409 - up, sign, sum);
      } else {
        bwd_dw<false, NA, NB>(pa, kBwdPlane, pb, lo_b, at_row, nullptr, 0, g, 0, sign, sum);
      }
    };
    // ---- dz of a layer's accumulator (values v, sample 16 m + 4 g + r) into
    // plane set `to`; the bias gradient in true units
    const auto dz_out = [&](float (&v)[4][4], unsigned int bits, int to, int l, float sz) {
      [[maybe_unused]] float largest = 0.0f;
      float sum = 0.0f;   // the chunk's bias gradient: fewer roundings at the total's size
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        f32x4 u = {1.0f, 1.0f, 1.0f, 1.0f};
        if constexpr (F16) u = *reinterpret_cast<const f32x4*>(&S.unit[16 * m + 4 * g]);
        u32x2 hi, lo;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v[m][r] = (bits >> (4 * m + r)) & 1u ? v[m][r] : 0.0f;
          sum = F16 ? __fmaf_rn(v[m][r], u[r], sum) : sum + v[m][r];
          if constexpr (F16) largest = fmaxf(largest, fabsf(v[m][r]));
        }
        asm volatile("" : "+v"(sum));
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          unsigned int hw, lw;
          parts2<F16>(v[m][2 * p], v[m][2 * p + 1], sz, sz, hw, lw);
          hi[p] = hw;
          lo[p] = lw;
        }
        *reinterpret_cast<u32x2*>(&S.t[to][at_out[m]]) = hi;
        *reinterpret_cast<u32x2*>(&S.t[to][kBwdPlane + at_out[m]]) = lo;
        tile_fence();
      }
      gb[l] = gb[l] + sum;
      if constexpr (F16) {
        const int m = row_max15(__float_as_int(largest));
        if (c == 15) S.dz_top[l][w][g] = short(m >> 16);
      }
    };
    // ---- dz2 = mask (W_head^T dl) in FP32, and dW_head
    {
      float v[4][4];
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float4 d = *reinterpret_cast<const float4*>(S.dl[16 * m + 4 * g + r]);
          v[m][r] = __fmaf_rn(wh[3], d.w, __fmaf_rn(wh[2], d.z, __fmaf_rn(wh[1], d.y, wh[0] * d.x)));
          if (r == 3) tile_fence();
        }
      dz_out(v, mask[2], 3, 2, F16 ? f16_scale(ez[0]) : 1.0f);
    }
    if constexpr (F16) {
      // in FP32 on the vector unit: lane (g, c) adds its 16 samples of feature
      // c, for the four logits in gh.  A logit's gradients can lie far below
      // its sample's largest, which is what the parts' scale would follow
      const unsigned short* ph = &S.t[2][16 * w * kBwdRow + bwd_at(c, 16 * g)];
      f32x4 sum = zero4;   // the chunk's: fewer roundings at the total's size
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const f16x8 h = __builtin_bit_cast(f16x8, lds128(ph + 8 * q));
        const f16x8 l = __builtin_bit_cast(f16x8, lds128(ph + 8 * q + kBwdPlane));
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int k = 16 * g + 8 * q + i;
          // the sample's unit over h2's scale (a power of two: its inverse)
          const float f = S.unit[k] * __int_as_float((254 << 23) - __float_as_int(S.scale[2][k]));
          const float x = __fmaf_rn(float(h[i]), f, float(l[i]) * f);
          const float4 d = *reinterpret_cast<const float4*>(S.dl[k]);
          sum[0] = __fmaf_rn(d.x, x, sum[0]);
          sum[1] = __fmaf_rn(d.y, x, sum[1]);
          sum[2] = __fmaf_rn(d.z, x, sum[2]);
          sum[3] = __fmaf_rn(d.w, x, sum[3]);
        }
        tile_fence();
      }
      gh = gh + sum;
    } else {
      f32x4 ghc = zero4;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        // dl of logit c (lanes c < 4) for samples 32 ks + 8 g + i
        unsigned int hw[4], lw[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          float v[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) v[k] = c < 4 ? S.dl[32 * ks + 8 * g + 2 * p + k][c & 3] : 0.0f;
          parts2<F16>(v[0], v[1], 1.0f, 1.0f, hw[p], lw[p]);
        }
        const unsigned short* pb = &S.t[2][16 * w * kBwdRow + at_row[ks]];
        ghc = mm16x3<F16>(u32x4{hw[0], hw[1], hw[2], hw[3]}, u32x4{lw[0], lw[1], lw[2], lw[3]},
                          lds128(pb), lds128(pb + kBwdPlane), ghc);
        tile_fence();
      }
      gh = gh + ghc;
    }
    asm volatile("" : "+v"(gh));
    __syncthreads();
    if (threadIdx.x < kBwdChunk) S.top0[threadIdx.x] = 0;

    const int row2 = 32 * (w & 3) * kBwdRow, col2 = 64 * (w >> 2) * kBwdRow;
    // ---- dW_2 (dz2 x h1); dz1 = mask (W_2^T dz2) into h2's planes
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[m] = zero4;
    bwd_layer<F16, 4>(S.t[3], at_tr, kBwdPlane, f, acc);
    f.load(F + 128 * (T::X_THIDDEN + w * T::KXH), lane);
    {
      const float bk = F16 ? f16_unscale(ez[0]) * f16_unscale(ew[2]) : 1.0f;
      float v[4][4];
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[m][r] = F16 ? acc[m][r] * bk : acc[m][r];
      dz_out(v, mask[1], 2, 1, F16 ? f16_scale(ez[1]) : 1.0f);
    }
    weight_gradient(std::integral_constant<int, 2>{}, &S.t[3][row2], &S.t[1][col2], kBwdPlane, gw2);
    __syncthreads();
    // ---- dW_1 (dz1 x h0); dz0 = mask (W_1^T dz1) into dz2's planes
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[m] = zero4;
    bwd_layer<F16, 4>(S.t[2], at_tr, kBwdPlane, f, acc);
    // W_0^T: the input gradient's tile w & 1 (features) of samples 16 (w / 2)..
    f.load(F + 128 * (T::X_T0 + (w & 1) * T::KXH), lane);
    {
      const float bk = F16 ? f16_unscale(ez[1]) * f16_unscale(ew[1]) : 1.0f;
      float v[4][4];
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[m][r] = F16 ? acc[m][r] * bk : acc[m][r];
      dz_out(v, mask[0], 3, 0, F16 ? f16_scale(ez[2]) : 1.0f);
    }
    weight_gradient(std::integral_constant<int, 1>{}, &S.t[2][row2], &S.t[0][col2], kBwdPlane, gw1);
    __syncthreads();
    // ---- dW_0 (dz0 x features) and the input gradient W_0^T dz0, whose
    // products run as W X so that a lane holds 4 features of a sample
    {
      const int m = w >> 1;
      const int at_m = bwd_at(4 * g + (c >> 2), 16 * m + 4 * (c & 3));
      f32x4 d = zero4;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) {
        const unsigned short* p = &S.t[3][at_m + kt * 32 * kBwdRow];
        d = mm16x3<F16>(f.h[kt], f.l[kt], lds_tr(p), lds_tr(p + kBwdPlane), d);
      }
      const int i = 16 * m + c;
      if constexpr (F16) d = (d * (f16_unscale(ez[2]) * f16_unscale(ew[0]))) * S.unit[i];
      if (s0 + i < M)
        *reinterpret_cast<f32x4*>(demb + (s0 + i) * D + 16 * (w & 1) + 4 * g) = d;
    }
    weight_gradient(std::integral_constant<int, 0>{}, &S.t[3][16 * w * kBwdRow], S.x0, kBwdPlane0, gw0);
    __syncthreads();
  }

  // ---- the block's partial sums, in torch order
  float* P = partial + int64_t(blockIdx.x) * T::PARAMS;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int64_t o = int64_t(32 * (w & 3) + 16 * a + 4 * g + r) * H + 64 * (w >> 2) + 16 * b + c;
        P[T::P_LAYER1 + o] = gw1[a][b][r];
        P[T::P_LAYER1 + int64_t(H) * H + H + o] = gw2[a][b][r];
      }
#pragma unroll
    for (int b = 0; b < 2; ++b)
      P[T::P_W0 + int64_t(16 * w + 4 * g + r) * D + 16 * b + c] = gw0[0][b][r];
    if constexpr (F16) {   // a lane group's samples each
      gh[r] = gh[r] + __shfl_xor(gh[r], 16, 64);
      gh[r] = gh[r] + __shfl_xor(gh[r], 32, 64);
    }
    if (g == 0) P[T::P_HEAD + int64_t(r) * H + 16 * w + c] = gh[r];
  }
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    float v = gb[l];
    v = v + __shfl_xor(v, 16, 64);
    v = v + __shfl_xor(v, 32, 64);
    const int64_t at = l == 0 ? T::P_B0 : T::P_LAYER1 + (l - 1) * (int64_t(H) * H + H) + int64_t(H) * H;
    if (g == 0) P[at + 16 * w + c] = v;
  }
  // the head's bias: waves 0-3 hold their samples' sums (lanes c < 4)
  ghb = ghb + __shfl_xor(ghb, 16, 64);
  ghb = ghb + __shfl_xor(ghb, 32, 64);
  if (w < 4 && lane < 4) S.dl[w][lane] = ghb;
  __syncthreads();
  if (threadIdx.x < 4)
    P[T::P_HEAD + 4 * H + threadIdx.x] =
        ((S.dl[0][threadIdx.x] + S.dl[1][threadIdx.x]) + S.dl[2][threadIdx.x]) + S.dl[3][threadIdx.x];
  if (F16 && threadIdx.x == 0) flags[blockIdx.x] = flagged;
}

// dparams[p] = the sum over blocks of partial[b][p], in a fixed order: lane
// group j of a block's 16 adds blocks j, j + 16, ..., four loads in flight, and
// the 16 sums are added in order.  nb16 partials, then nb32 more where one of
// the nb16 flags is set.
// A thread per parameter waited for nb loads one by one: 61 us for 256
// partials, now 16.
constexpr int kSumCols = 16;   // parameters per block
__global__ __launch_bounds__(256) void sum_partials_kernel(const float* __restrict__ partial,
                                                           int nb16, int nb32, int64_t P,
                                                           const int32_t* __restrict__ flags,
                                                           float* __restrict__ dparams) {
  __shared__ float sums[16][kSumCols];
  int flagged = 0;
  if (flags)
    for (int i = threadIdx.x; i < nb16; i += 256) flagged |= flags[i];
  const int nb = nb16 + (__syncthreads_or(flagged) ? nb32 : 0);
  const int j = threadIdx.x / kSumCols, q = threadIdx.x % kSumCols;
  const int64_t p = int64_t(blockIdx.x) * kSumCols + q;
  float acc = 0.0f;
  if (p < P) {
    int b = j;
    for (; b + 48 < nb; b += 64) {
      const float v0 = partial[int64_t(b) * P + p], v1 = partial[int64_t(b + 16) * P + p];
      const float v2 = partial[int64_t(b + 32) * P + p], v3 = partial[int64_t(b + 48) * P + p];
      acc = (((acc + v0) + v1) + v2) + v3;
    }
    for (; b < nb; b += 16) acc = acc + partial[int64_t(b) * P + p];
  }
  sums[j][q] = acc;
  __syncthreads();
  if (j == 0 && p < P) {
#pragma unroll
    for (int k = 1; k < 16; ++k) acc = acc + sums[k][q];
    dparams[p] = acc;
  }
}

// The layers' weights and biases, device pointers.
struct TrainLayers {
  const float* w[8];
  const float* b[8];
};

// Layer l's weights are positions start[l] .. start[l + 1] - 1 of [0, W_0
// flat, W_1 flat, ...].
struct SplitLayers {
  TrainLayers net;
  int64_t start[9];
  int H, L;
};

// Elements of the split-BF16 fragments, at the positions index[] gives (the
// forward kernel's, then the backward's): per 512 their hi parts bf16(w), then
// their lo parts bf16(w - hi); the biases in one row, the head's 4 padded to
// 16; and count.  One launch: the copies, conversions and differences were 16
// torch launches in every training step.
__global__ __launch_bounds__(256) void split_pack_kernel(SplitLayers s,
                                                         const int64_t* __restrict__ index,
                                                         int64_t n_forward, int64_t n_backward,
                                                         __bf16* __restrict__ forward,
                                                         __bf16* __restrict__ backward,
                                                         float* __restrict__ bias, int count,
                                                         int32_t* __restrict__ count_dev) {
  int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i == 0) *count_dev = count;
  if (i < n_forward + n_backward) {
    const int64_t p = index[i];
    float w = 0.0f;
    for (int l = 0; l <= s.L; ++l)
      if (p >= s.start[l] && p < s.start[l + 1]) w = s.net.w[l][p - s.start[l]];
    __bf16* out = i < n_forward ? forward : backward;
    if (i >= n_forward) i -= n_forward;
    const __bf16 hi = __bf16(w);
    out[(i >> 9) * 1024 + (i & 511)] = hi;
    out[(i >> 9) * 1024 + 512 + (i & 511)] = __bf16(w - float(hi));
    return;
  }
  i -= n_forward + n_backward;
  const int64_t hidden = int64_t(s.L) * s.H;
  if (i < hidden)
    bias[i] = s.net.b[i / s.H][i % s.H];
  else if (i < hidden + 16)
    bias[i] = i < hidden + 4 ? s.net.b[s.L][i - hidden] : 0.0f;
}

// Block l: layer l's largest |w|, row sum |w|, column sum |w| and b, the last 0
// at least (not finite where a value is not; a bias of -inf is a unit switched
// off).  The largest |w| is infinite, too, where one scale does not do for the
// layer (kF16Spread).
template <int D, int H, int L>
__global__ __launch_bounds__(1024) void mlp_stats_kernel(TrainLayers net,
                                                         float* __restrict__ stats) {
  __shared__ int best[4], least;
  __shared__ float cols[16][H], tops[16][H];   // each wave's column sums and maxima
  const int l = blockIdx.x, rows = l < L ? H : 4, in = l == 0 ? D : H;
  const float* W = net.w[l];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (threadIdx.x < 4) best[threadIdx.x] = 0;
  if (threadIdx.x == 0) least = 0x7F800000;
  __syncthreads();
  // |x| as integer bits order as the values do, NaN and infinity on top
  const auto up = [&](int k, float v) {
    int m = __float_as_int(v) & 0x7FFFFFFF;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) m = max(m, __shfl_xor(m, d, 64));
    if (lane == 0) atomicMax(&best[k], m);
  };
  // a wave's rows, all loads in flight
  constexpr int R = H / 16;
  float v[R][H / 64];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int q = 0; q < H / 64; ++q) {
      const int r = wave + 16 * i, k = lane + 64 * q;
      v[i][q] = r < rows && k < in ? fabsf(W[r * in + k]) : 0.0f;
    }
  float widest = 0.0f;
  int top = 0;
  float mine[H / 64] = {};
  int most[H / 64] = {};
#pragma unroll
  for (int i = 0; i < R; ++i) {
    float sum = 0.0f;
    int row = 0;
#pragma unroll
    for (int q = 0; q < H / 64; ++q) {
      row = max(row, __float_as_int(v[i][q]));
      most[q] = max(most[q], __float_as_int(v[i][q]));
      mine[q] += v[i][q];
      sum += v[i][q];
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, 64);
    row = wave_max(row);
    widest = __int_as_float(max(__float_as_int(widest), __float_as_int(sum) & 0x7FFFFFFF));
    top = max(top, row);
    if (lane == 0 && row != 0) atomicMin(&least, row);
  }
  up(1, widest);
  up(0, __int_as_float(top));
#pragma unroll
  for (int q = 0; q < H / 64; ++q) {
    cols[wave][lane + 64 * q] = mine[q];
    tops[wave][lane + 64 * q] = __int_as_float(most[q]);
  }
  float b = 0.0f;
  for (int i = threadIdx.x; i < rows; i += 1024) {
    const float bi = net.b[l][i];   // one below 0 only lowers its unit
    b = __int_as_float(max(__float_as_int(b), bi < 0.0f ? 0 : __float_as_int(bi) & 0x7FFFFFFF));
  }
  up(3, b);
  __syncthreads();
  // the waves' sums in order: the sums choose scales, so their last bits must
  // not depend on timing
  float col = 0.0f;
  if (threadIdx.x < H) {
    int most = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      col += cols[w][threadIdx.x];
      most = max(most, __float_as_int(tops[w][threadIdx.x]));
    }
    if (most != 0) atomicMin(&least, most);
  }
  up(2, col);
  __syncthreads();
  // row and column sums a little above their rounding
  if (threadIdx.x < 4) {
    float v = __int_as_float(best[threadIdx.x]);
    if (threadIdx.x == 0 && __int_as_float(least) < v * kF16Spread) v = INFINITY;
    stats[threadIdx.x * (L + 1) + l] = threadIdx.x == 1 || threadIdx.x == 2 ? v * 1.001f : v;
  }
}

// Element e (of 64 lanes x 8) of the 16-bit kernels' fragment f, in the order
// of TrainDims::X_* and then the head's forward fragments: lane (g, c) of
// fragment (mt, kt) holds W[16 mt + c][32 kt + 4 g + i, + 16 for i >= 4] of its
// layer, or of the layer's transpose.
template <int D, int H, int L>
__device__ __forceinline__ float fragment_value(const TrainLayers& net, int f, int lane, int i,
                                                int* layer) {
  using T = TrainDims<D, H, L>;
  bool transposed = false;
  int l, n, KT;
  if (f < T::X_HIDDEN) {
    l = 0, n = f, KT = T::KX0;
  } else if (f < T::X_T0) {
    n = f - T::X_HIDDEN, l = 1 + n / (T::MT * T::KXH), n %= T::MT * T::KXH, KT = T::KXH;
  } else if (f < T::X_THIDDEN) {
    transposed = true, l = 0, n = f - T::X_T0, KT = T::KXH;
  } else if (f < T::X_FRAGS) {
    transposed = true;
    n = f - T::X_THIDDEN, l = 1 + n / (T::MT * T::KXH), n %= T::MT * T::KXH, KT = T::KXH;
  } else {
    l = L, n = f - T::X_FRAGS, KT = T::KXH;
  }
  *layer = l;
  const int g = lane >> 4, c = lane & 15;
  const int row = 16 * (n / KT) + c, col = 32 * (n % KT) + 4 * g + (i & 3) + (i >= 4 ? 16 : 0);
  const int in = l == 0 ? D : H;
  if (transposed) return net.w[l][col * in + row];
  return l == L && row >= 4 ? 0.0f : net.w[l][row * in + col];
}

// Packs the weights: the FP32 fragments of TrainDims (forward, then
// transposed), the biases, and the FP16 fragments scaled by the layers' power
// of two (stats: mlp_stats_kernel's, in `packed`).  Thread per float.
//   forward [ceil(Hout/16)][Hin/4][64], lane (g, c) of fragment (mt, 4t + i)
//     = W[16 mt + c][16 t + 4 g + i] (0 past Hout);
//   transposed [Hin/16][Hout/4][64], lane (g, c) of fragment (mt, 4t + i)
//     = W[16 t + 4 g + i][16 mt + c];
//   transposed head [Hin/16][64], lane (g, c) of fragment mt = W[g][16 mt + c].
// One launch (after the stats') where each layer and form and each bias took
// one of its own: 25 -> 17 us per call, 2 launches instead of 12.
template <int D, int H, int L>
__global__ __launch_bounds__(256) void mlp_pack_kernel(TrainLayers net,
                                                       float* __restrict__ packed) {
  using T = TrainDims<D, H, L>;
  const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (p >= T::PACKED || (p >= T::STATS_BASE && p < T::F16_BASE)) return;
  if (p >= T::F16_BASE) {
    // pairs of parts: thread = (fragment, part, lane, pair)
    const int64_t q = p - T::F16_BASE;
    const int f = int(q / 512), part = int(q / 256) & 1, lane = int(q / 4) & 63, i = 2 * int(q & 3);
    int l;
    const float a = fragment_value<D, H, L>(net, f, lane, i, &l);
    const float b = fragment_value<D, H, L>(net, f, lane, i + 1, &l);
    const float s = f16_scale(min(f16_exponent(packed[T::STATS_BASE + l]), 254));
    f16x2 hi, lo;
    f16_split2(a, b, s, s, hi, lo);
    packed[p] = __builtin_bit_cast(float, part ? lo : hi);
    return;
  }
  if (p >= T::BIAS_BASE) {
    const int q = int(p - T::BIAS_BASE), l = min(q / H, L);
    packed[p] = net.b[l][q - l * H];
    return;
  }
  const bool transposed = p >= T::T_BASE;
  const int64_t q = transposed ? p - T::T_BASE : p;
  const int lane = int(q & 63), g = lane >> 4, c = lane & 15;
  int n = int(q >> 6), l, KT;
  if (!transposed) {
    if (n < T::F_HIDDEN) {
      l = 0, KT = T::KT0;
    } else {
      n -= T::F_HIDDEN, l = min(1 + n / (T::MT * T::KTH), L), n -= (l - 1) * T::MT * T::KTH;
      KT = T::KTH;
    }
    const int row = 16 * (n / KT) + c, kt = n % KT, in = l == 0 ? D : H;
    packed[p] = l == L && row >= 4 ? 0.0f : net.w[l][row * in + 16 * (kt >> 2) + 4 * g + (kt & 3)];
    return;
  }
  if (n >= T::T_HEAD) {
    packed[p] = net.w[L][g * H + 16 * (n - T::T_HEAD) + c];
    return;
  }
  if (n < T::T_HIDDEN) {
    l = 0;
  } else {
    n -= T::T_HIDDEN, l = 1 + n / (T::MT * T::KTH), n %= T::MT * T::KTH;
  }
  const int mt = n / T::KTH, kt = n % T::KTH, in = l == 0 ? D : H;
  packed[p] = net.w[l][(16 * (kt >> 2) + 4 * g + (kt & 3)) * in + 16 * mt + c];
}

template <int D, int H, int L>
int pack_impl(const float* const* weights, const float* const* biases, float* packed,
              hipStream_t st) {
  using T = TrainDims<D, H, L>;
  static_assert(L + 1 <= 8, "TrainLayers");
  TrainLayers net{};
  for (int l = 0; l <= L; ++l) {
    net.w[l] = weights[l];
    net.b[l] = biases[l];
  }
  hipLaunchKernelGGL((mlp_stats_kernel<D, H, L>), dim3(L + 1), dim3(1024), 0, st, net,
                     packed + T::STATS_BASE);
  if (check_launch("mlp_train_stats") != NSVF_OK) return NSVF_ELAUNCH;
  hipLaunchKernelGGL((mlp_pack_kernel<D, H, L>), dim3(unsigned(ceil_div(T::PACKED, 256))),
                     dim3(256), 0, st, net, packed);
  return check_launch("mlp_train_pack");
}

// Blocks (and partials) of the 16-bit backward kernel and of the FP32 one.
int backward_blocks(int64_t M, int64_t chunk) {
  return int(std::max<int64_t>(1, std::min<int64_t>(ceil_div(M, chunk), kMaxTrainBlocks)));
}

constexpr size_t kBackwardLds = size_t(2) * kTrainChunk * kLdsRow * sizeof(float);

bool train_shape_ok(int D, int H, int L) { return D == 32 && H == 128 && L == 3; }

}  // namespace
}  // namespace nsvf

using namespace nsvf;

extern "C" {

int nsvf_mlp_train_supported(int D, int H, int L) { return train_shape_ok(D, H, L) ? 1 : 0; }

int64_t nsvf_mlp_train_packed_floats(int D, int H, int L) {
  if (!train_shape_ok(D, H, L)) return -1;
  return TrainDims<32, 128, 3>::PACKED;
}

int64_t nsvf_mlp_train_param_floats(int D, int H, int L) {
  if (!train_shape_ok(D, H, L)) return -1;
  return TrainDims<32, 128, 3>::PARAMS;
}

int64_t nsvf_mlp_train_partial_floats(int D, int H, int L, int64_t M) {
  if (!train_shape_ok(D, H, L) || M < 0) return -1;
  // the partial sums of the 16-bit kernel's blocks and of the FP32 one's, the
  // first's flags and the chunks'
  const int64_t nb = backward_blocks(M, kBwdChunk);
  constexpr int64_t P = TrainDims<32, 128, 3>::PARAMS;
  return M == 0 ? nb * P
                : (nb + backward_blocks(M, kTrainChunk)) * P + nb + ceil_div(M, kBwdChunk);
}

int nsvf_mlp_split_pack(int D, int H, int L, const float* const* weights,
                        const float* const* biases, const int64_t* index, int64_t n_forward,
                        int64_t n_backward, void* forward, void* backward, float* bias, int count,
                        int32_t* count_dev, void* stream) {
  clear_error();
  if (D <= 0 || H <= 0 || L <= 0 || L > 7 || n_forward < 0 || n_backward < 0 ||
      n_forward % 512 != 0 || n_backward % 512 != 0)
    return set_error(NSVF_EINVAL, "mlp_split_pack: bad size");
  if (!weights || !biases || !index || !bias || !count_dev || (n_forward > 0 && !forward) ||
      (n_backward > 0 && !backward))
    return set_error(NSVF_EINVAL, "mlp_split_pack: null pointer");
  for (int l = 0; l <= L; ++l)
    if (!weights[l] || !biases[l]) return set_error(NSVF_EINVAL, "mlp_split_pack: layer %d null", l);
  SplitLayers net;
  int64_t at = 1;
  for (int l = 0; l <= L; ++l) {
    net.net.w[l] = weights[l];
    net.net.b[l] = biases[l];
    net.start[l] = at;
    at += int64_t(l < L ? H : 4) * (l == 0 ? D : H);
  }
  net.start[L + 1] = at;
  net.H = H;
  net.L = L;
  const int64_t n = n_forward + n_backward + L * H + 16;
  hipLaunchKernelGGL(split_pack_kernel, dim3(unsigned(ceil_div(n, 256))), dim3(256), 0,
                     as_stream(stream), net, index, n_forward, n_backward,
                     static_cast<__bf16*>(forward), static_cast<__bf16*>(backward), bias, count,
                     count_dev);
  return check_launch("mlp_split_pack");
}

int nsvf_mlp_train_pack(int D, int H, int L, const float* const* weights,
                        const float* const* biases, float* packed, void* stream) {
  clear_error();
  if (!train_shape_ok(D, H, L))
    return set_error(NSVF_EINVAL, "mlp_train_pack: shape D=%d H=%d L=%d (built: 32, 128, 3)", D,
                     H, L);
  if (!weights || !biases || !packed) return set_error(NSVF_EINVAL, "mlp_train_pack: null");
  for (int l = 0; l <= L; ++l)
    if (!weights[l] || !biases[l]) return set_error(NSVF_EINVAL, "mlp_train_pack: layer %d null", l);
  return pack_impl<32, 128, 3>(weights, biases, packed, as_stream(stream));
}

int nsvf_mlp_train_forward(int D, int H, int L, const float* packed, const float* emb, int64_t M,
                           float* out, void* stream) {
  clear_error();
  if (!train_shape_ok(D, H, L))
    return set_error(NSVF_EINVAL, "mlp_train_forward: shape D=%d H=%d L=%d (built: 32, 128, 3)",
                     D, H, L);
  if (M < 0) return set_error(NSVF_EINVAL, "mlp_train_forward: M=%lld", static_cast<long long>(M));
  if (M == 0) return NSVF_OK;
  if (!packed || !emb || !out) return set_error(NSVF_EINVAL, "mlp_train_forward: null pointer");
  using Mlp = F16Mlp<32, 128, 3>;
  static_assert(Mlp::fits(), "weights staged in LDS");
  const int64_t tiles = ceil_div(M, kF16Samples);
  // one block per CU (the weights fill its LDS), fewer for fewer tiles
  const unsigned grid = unsigned(std::min<int64_t>(ceil_div(tiles, kF16Waves), kMaxTrainBlocks));
  hipLaunchKernelGGL((mlp_train_forward_kernel<32, 128, 3>), dim3(grid), dim3(64 * kF16Waves),
                     Mlp::LDS_BYTES, as_stream(stream), emb, M, packed, out);
  return check_launch("mlp_train_forward");
}

int64_t nsvf_mlp_train_x3_frags(int D, int H, int L) {
  if (!train_shape_ok(D, H, L)) return -1;
  return TrainDims<32, 128, 3>::X_FRAGS;
}

static int train_backward(const char* name, int D, int H, int L, const float* packed,
                          const int16_t* x3w, const float* emb, int64_t M, const float* dout,
                          float* demb, float* partial, int64_t partial_floats, float* dparams,
                          void* stream) {
  if (!train_shape_ok(D, H, L))
    return set_error(NSVF_EINVAL, "%s: shape D=%d H=%d L=%d (built: 32, 128, 3)", name, D, H, L);
  if (M < 0) return set_error(NSVF_EINVAL, "%s: M=%lld", name, static_cast<long long>(M));
  if (!packed || !partial || !dparams || (M > 0 && (!emb || !dout || !demb)))
    return set_error(NSVF_EINVAL, "%s: null pointer", name);
  using T = TrainDims<32, 128, 3>;
  const int64_t need = nsvf_mlp_train_partial_floats(D, H, L, M);
  if (partial_floats < need)
    return set_error(NSVF_EINVAL, "%s: partial buffer of %lld floats, %lld needed", name,
                     static_cast<long long>(partial_floats), static_cast<long long>(need));
  hipStream_t st = as_stream(stream);
  const int nb = backward_blocks(M, kBwdChunk), nb32 = backward_blocks(M, kTrainChunk);
  float* partial32 = partial + int64_t(nb) * T::PARAMS;
  int32_t* flags = x3w || M == 0 ? nullptr
                                 : reinterpret_cast<int32_t*>(partial32 + int64_t(nb32) * T::PARAMS);
  if (x3w || M == 0) {
    hipLaunchKernelGGL((mlp_train_backward_kernel<32, 128, 3, false>), dim3(nb), dim3(kBwdBlock),
                       sizeof(BwdLds), st, emb, M, packed, reinterpret_cast<const u32x4*>(x3w),
                       dout, demb, partial, flags, nullptr);
    if (check_launch(name) != NSVF_OK) return NSVF_ELAUNCH;
  } else {
    int32_t* chunk_flags = flags + nb;
    hipLaunchKernelGGL((mlp_train_backward_kernel<32, 128, 3, true>), dim3(nb), dim3(kBwdBlock),
                       sizeof(BwdLds), st, emb, M, packed,
                       reinterpret_cast<const u32x4*>(packed + T::F16_BASE), dout, demb, partial,
                       flags, chunk_flags);
    if (check_launch(name) != NSVF_OK) return NSVF_ELAUNCH;
    hipLaunchKernelGGL((mlp_train_backward_f32_kernel<32, 128, 3>), dim3(nb32), dim3(kTrainBlock),
                       kBackwardLds, st, emb, M, packed, dout, demb, partial32, flags, nb,
                       chunk_flags);
    if (check_launch(name) != NSVF_OK) return NSVF_ELAUNCH;
  }
  hipLaunchKernelGGL(sum_partials_kernel, dim3(unsigned(ceil_div(T::PARAMS, kSumCols))), dim3(256),
                     0, st, partial, nb, nb32, T::PARAMS, flags, dparams);
  return check_launch("mlp_train_sum_partials");
}

int nsvf_mlp_train_backward(int D, int H, int L, const float* packed, const float* emb,
                            int64_t M, const float* dout, float* demb, float* partial,
                            int64_t partial_floats, float* dparams, void* stream) {
  clear_error();
  return train_backward("mlp_train_backward", D, H, L, packed, nullptr, emb, M, dout, demb,
                        partial, partial_floats, dparams, stream);
}

int nsvf_mlp_train_backward_x3(int D, int H, int L, const float* packed, const int16_t* x3w,
                               const float* emb, int64_t M, const float* dout, float* demb,
                               float* partial, int64_t partial_floats, float* dparams,
                               void* stream) {
  clear_error();
  if (!x3w || reinterpret_cast<uintptr_t>(x3w) % 16 != 0)
    return set_error(NSVF_EINVAL, "mlp_train_backward_x3: fragments null or not 16-byte aligned");
  return train_backward("mlp_train_backward_x3", D, H, L, packed, x3w, emb, M, dout, demb,
                        partial, partial_floats, dparams, stream);
}

}  // extern "C"
