// Kernels of the learned proposer: bf16 copies, batched forward, gradients (forward and backward on the
// MFMA units, four waves of a block on 64 rows each at a time, one partial gradient per block), and the
// reduction of the partial gradients with an Adam step.
#include <hip/hip_runtime.h>

#include "mlp_dev.h"

namespace bsx {
namespace mlp {

namespace {

__global__ void to_bf16_kernel(const float* w, uint16_t* wb, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) wb[i] = to_bf16(w[i]);
}

// ---- Activations that stay in registers -------------------------------------------------------------
// The products run transposed, hidden units by rows: a lane's accumulator of a 32x32 tile holds 16 units of one
// row (unit 8 (j / 4) + 4 (l / 32) + j % 4, row l % 32), which, rounded to bf16 eight at a time, is the next
// product's B operand as it stands, if the weights' operand takes its k index in the same order (unit_of). So
// no activation passes through LDS on the way, and a lane applies silu to its own accumulators.
// v_mfma_f32_32x32x16_bf16: lane l supplies A[l % 32][8 (l / 32) + i] and B[8 (l / 32) + i][l % 32], i = 0..7.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
typedef bf16x8 bf16x8_lds __attribute__((may_alias));  // eight 16-bit words of LDS read as one operand

__device__ __forceinline__ f32x16 mma(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// The hidden unit of element i of k-chunk c for the lanes of half h: the unit of accumulator element 8 (c % 2) + i of
// tile c / 2.
__host__ __device__ constexpr int unit_of(int c, int h, int i) { return 16 * c + 8 * (i >> 2) + 4 * h + (i & 3); }
constexpr bool unit_of_matches_accumulators() {
  for (int c = 0; c < 4; ++c)
    for (int h = 0; h < 2; ++h)
      for (int i = 0; i < 8; ++i)
        if (unit_of(c, h, i) != 32 * (c >> 1) + acc_row_of(8 * (c & 1) + i, h)) return false;
  return true;
}
static_assert(unit_of_matches_accumulators());

__device__ __forceinline__ __bf16 bits_bf16(uint16_t u) { return __builtin_bit_cast(__bf16, u); }

// z sigma(z) and sigma by the hardware exponential and reciprocal (an ulp each: far inside the rounding to
// bf16 that follows).
__device__ __forceinline__ float sigmoid_fast(float z) { return __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }

// The operand of W1 and W2 of one wave: W1^T (two tiles of units, one k-chunk of features) and W2^T (two tiles of
// units, four k-chunks).
struct ForwardWeights {
  bf16x8 w1[2], w2[2][4];
};

__device__ __forceinline__ void load_forward(ForwardWeights& f, const WeightsLds& w) {
  const int l = threadIdx.x & 63, m = l & 31, h = l >> 5;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 8; ++i) f.w1[t][i] = bits_bf16(w.w1[(8 * h + i) * kS16 + t * 32 + m]);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int i = 0; i < 8; ++i) f.w2[t][c][i] = bits_bf16(w.w2[unit_of(c, h, i) * kS16 + t * 32 + m]);
}

// load_weights for a block of 256 threads: 16-byte vectors, every load under way before the first is stored.
__device__ __forceinline__ void load_weights_256(WeightsLds& s, const uint16_t* wb, const float* w) {
  static_assert(kOffW1 % 8 == 0 && kOffW2 % 8 == 0 && kS16 % 8 == 0 && kHid == 64 && kIn * kHid / 8 <= 256);
  const int tid = threadIdx.x;
  const uint4* w2 = reinterpret_cast<const uint4*>(wb + kOffW2);
  const uint4* w1 = reinterpret_cast<const uint4*>(wb + kOffW1);
  const uint4 a = w2[tid], b = w2[tid + 256];
  uint4 c = {0, 0, 0, 0};
  if (tid < kIn * kHid / 8) c = w1[tid];
  float f = 0.0f;  // b1, b2, w3 (its bf16 value) and b3, 64 threads each
  if (tid < 64) f = w[kOffB1 + tid];
  else if (tid < 128) f = w[kOffB2 + tid - 64];
  else if (tid < 192) f = from_bf16(wb[kOffW3 + tid - 128]);
  else if (tid == 192) f = w[kOffB3];
  *reinterpret_cast<uint4*>(s.w2 + (tid >> 3) * kS16 + (tid & 7) * 8) = a;
  *reinterpret_cast<uint4*>(s.w2 + (32 + (tid >> 3)) * kS16 + (tid & 7) * 8) = b;
  if (tid < kInPad * kHid / 8) *reinterpret_cast<uint4*>(s.w1 + (tid >> 3) * kS16 + (tid & 7) * 8) = c;
  if (tid < 64) s.b1[tid] = f;
  else if (tid < 128) s.b2[tid - 64] = f;
  else if (tid < 192) s.w3[tid - 128] = f;
  else if (tid == 192) s.b3 = f;
  __syncthreads();
}

// This lane's eight features of row `row` as the B operand (features 12 .. 15 and rows past n zero). kWide: x is
// 16-byte aligned, so that a row's twelve floats are three aligned vectors.
template <bool kWide>
__device__ __forceinline__ bf16x8 load_features(const float* x, int64_t row, bool valid) {
  const int h = (threadIdx.x & 63) >> 5;
  f32x8 v = {};
  if (valid) {
    const float* r = x + row * kIn + 8 * h;
    if constexpr (kWide) {
      const float4 a = *reinterpret_cast<const float4*>(r);
      v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
      if (h == 0) {
        const float4 b = *reinterpret_cast<const float4*>(r + 4);
        v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (8 * h + i < kIn) v[i] = r[i];
    }
  }
  return __builtin_convertvector(v, bf16x8);
}

// k-chunk c of a tile pair's values, rounded to bf16.
__device__ __forceinline__ bf16x8 chunk(const f32x16* v, int c) {
  f32x8 e;
#pragma unroll
  for (int i = 0; i < 8; ++i) e[i] = v[c >> 1][8 * (c & 1) + i];
  return __builtin_convertvector(e, bf16x8);
}

// z + b for a tile pair's pre-activations: lane half h's units of tile t, four at a time.
__device__ __forceinline__ void add_bias(f32x16* z, const float* b) {
  const int h = (threadIdx.x & 63) >> 5;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(b + t * 32 + 8 * q + 4 * h);
      z[t][4 * q] += v.x;
      z[t][4 * q + 1] += v.y;
      z[t][4 * q + 2] += v.z;
      z[t][4 * q + 3] += v.w;
    }
}

// Pre-activations of both layers and the output of 32 rows (xb: their features); h1: the first layer's
// activations as the B operand.
__device__ __forceinline__ float forward_rows(const ForwardWeights& f, const WeightsLds& w, bf16x8 xb, f32x16* z1,
                                              bf16x8* h1, f32x16* z2) {
#pragma unroll
  for (int t = 0; t < 2; ++t) z1[t] = mma(f.w1[t], xb, f32x16{});
  add_bias(z1, w.b1);
  f32x16 a[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j) a[t][j] = z1[t][j] * sigmoid_fast(z1[t][j]);
#pragma unroll
  for (int c = 0; c < 4; ++c) h1[c] = chunk(a, c);
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    z2[t] = f32x16{};
#pragma unroll
    for (int c = 0; c < 4; ++c) z2[t] = mma(f.w2[t][c], h1[c], z2[t]);
  }
  add_bias(z2, w.b2);
  const int h = (threadIdx.x & 63) >> 5;
  float y = 0.0f;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 w3 = *reinterpret_cast<const float4*>(w.w3 + t * 32 + 8 * q + 4 * h);
      const float wv[4] = {w3.x, w3.y, w3.z, w3.w};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float z = z2[t][4 * q + r];
        y += static_cast<float>(static_cast<__bf16>(z * sigmoid_fast(z))) * wv[r];
      }
    }
  return y + __shfl_xor(y, 32) + w.b3;
}

// Bound by the activations on the VALU (128 exponentials and reciprocals a row against 20 MFMA per 64 rows): four
// waves a block, each 32 rows at a time, the weights in registers. 4 M rows: 0.18 ms (216 TFLOP/s); 1.35 ms with the
// operands gathered element by element from LDS and correctly rounded divisions.
template <bool kWide>
__global__ __launch_bounds__(256) void forward_kernel(const uint16_t* wb, const float* w, const float* x, int64_t n,
                                                      float* y) {
  __shared__ __align__(16) WeightsLds W;
  load_weights_256(W, wb, w);
  ForwardWeights f;
  load_forward(f, W);
  const int l = threadIdx.x & 63;
  const int64_t groups = (n + 31) / 32, stride = static_cast<int64_t>(gridDim.x) * 4;
  int64_t g = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  bf16x8 xb = load_features<kWide>(x, g * 32 + (l & 31), g * 32 + (l & 31) < n);
  for (; g < groups; g += stride) {
    const int64_t row = g * 32 + (l & 31), next = row + stride * 32;
    const bf16x8 xn = load_features<kWide>(x, next, next < n);  // the next rows' features, meanwhile
    f32x16 z1[2], z2[2];
    bf16x8 h1[4];
    const float out = forward_rows(f, W, xb, z1, h1, z2);
    if (l < 32 && row < n) y[row] = out;
    xb = xn;
  }
}

// Sum over the 32 lanes of a half of each of 32 values per lane: lane r of the half returns the sum of value r.
__device__ __forceinline__ float sum_scatter(float* v) {
  const int l = threadIdx.x & 31;
#pragma unroll
  for (int half = 16; half > 0; half >>= 1) {
    const bool upper = (l & half) != 0;
#pragma unroll
    for (int k = 0; k < half; ++k) {
      const float lo = v[k], hi = v[k + half];  // (both read: a chosen one would be an indexed read)
      v[k] = (upper ? hi : lo) + __shfl_xor(upper ? lo : hi, half);
    }
  }
  return v[0];
}

constexpr int kStepRows = 256;       // rows of a block's pass: 64 per wave
constexpr int kMaxPartials = 512;    // blocks of a gradient launch
constexpr int kRowStride = 72;       // of the transposed bf16 matrices (units by rows): 16-byte rows, no bank aliasing

// A wave's LDS: the transposed operands of the weight gradients (units by the wave's 64 rows); once they are
// consumed, its partial gradient.
struct GradLds {
  union {
    struct {
      uint16_t h1[kHid * kRowStride], dz2[kHid * kRowStride], dz1[kHid * kRowStride], xs[kIn * kRowStride];
    };
    float partial[kParams];
  };
};

// Gradients of (1 / batch) sum (y - t)^2, one partial gradient vector and squared error per block. Each wave runs
// 64 rows at a time through forward and backward with its activations in registers (dH1^T = W2 dZ2^T takes dZ2^T
// as the forward's products take theirs); only the weight gradients, which contract over the rows, read
// transposed copies from LDS, as 16-byte vectors. They are accumulated in registers over the block's rows and the
// four waves' sums added in order. A step of 65,536 rows (one pass of 256 blocks) takes 20.2 us, and 5.3 for the
// 256 partials' sum and Adam step; with operands gathered from LDS element by element and 1,024 partials of 64
// rows it took 47.5 and 51. Bound by the chain of one wave per SIMD.
template <bool kWide>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void gradients_kernel(const uint16_t* wb, const float* w, const float* x,
                                                           const float* target, int64_t n, float two_over_batch,
                                                           float* partial, float* loss_partial) {
  __shared__ __align__(16) WeightsLds W;
  __shared__ __align__(16) GradLds lds[4];
  load_weights_256(W, wb, w);
  const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63, col = l & 31, h = l >> 5;
  GradLds& S = lds[wave];
  ForwardWeights f;
  load_forward(f, W);
  // W2 as the backward product's operand (tile t of layer-1 units, k-chunk c of layer-2 units): two runs of four
  const auto w2_back = [&](int t, int c) {
    const uint16_t* r = W.w2 + (t * 32 + col) * kS16 + 16 * c + 4 * h;
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = bits_bf16(r[8 * (i >> 2) + (i & 3)]);
    return v;
  };
  f32x16 dw2[2][2] = {}, dw1[2] = {};  // tiles of W2 (layer-1 by layer-2 units) and of W1 (features by units)
  f32x4 db2[4] = {};  // 16 units a tile, the sum in every row
  float dw3 = 0.0f, db3 = 0.0f, se = 0.0f;  // dw3: of value col of the half (see sum_scatter)
  const u16x8 one = {0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80};
  const bf16x8 ones = __builtin_bit_cast(bf16x8, one);
  for (int64_t base = static_cast<int64_t>(blockIdx.x) * kStepRows; base < n;
       base += static_cast<int64_t>(gridDim.x) * kStepRows) {
    bf16x8 features[2];
    float targets[2];
    for (int b = 0; b < 2; ++b) {
      const int64_t row = base + wave * 64 + b * 32 + col;
      features[b] = load_features<kWide>(x, row, row < n);
      targets[b] = row < n ? target[row] : 0.0f;
    }
#pragma nounroll
    for (int b = 0; b < 2; ++b) {
      float sum[32];  // dy h2 of the lane's row and units
      const int at = b * 32 + col;  // the row's place among the wave's 64
      const int64_t row = base + wave * 64 + at;
      const bool valid = row < n;
      const bf16x8 xb = b == 0 ? features[0] : features[1];
      f32x16 z1[2], z2[2];
      bf16x8 h1[4], d2[4];
      const float y = forward_rows(f, W, xb, z1, h1, z2);
      const float e = valid ? y - (b == 0 ? targets[0] : targets[1]) : 0.0f;
      const float dy = e * two_over_batch;
      if (h == 0) {
        se += e * e;
        db3 += dy;
      }
      // dz2 = dy w3 silu'(z2), and the sum over the rows of dy h2 (in fp32)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int u = t * 32 + 8 * (j >> 2) + 4 * h + (j & 3);
          const float z = z2[t][j], s = sigmoid_fast(z);
          sum[t * 16 + j] = dy * static_cast<float>(static_cast<__bf16>(z * s));
          z2[t][j] = dy * W.w3[u] * (s * (1.0f + z * (1.0f - s)));
        }
      dw3 += sum_scatter(sum);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        d2[c] = chunk(z2, c);
        const u16x8 hb = __builtin_bit_cast(u16x8, h1[c]), db = __builtin_bit_cast(u16x8, d2[c]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int u = unit_of(c, h, i);
          S.h1[u * kRowStride + at] = hb[i];
          S.dz2[u * kRowStride + at] = db[i];
        }
      }
      // dh1^T = W2 dz2^T, dz1 = dh1 silu'(z1)
      f32x16 dh[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        dh[t] = f32x16{};
#pragma unroll
        for (int c = 0; c < 4; ++c) dh[t] = mma(w2_back(t, c), d2[c], dh[t]);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const float z = z1[t][j], s = sigmoid_fast(z);
          dh[t][j] *= s * (1.0f + z * (1.0f - s));
        }
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const bf16x8 d1 = chunk(dh, c);
        const u16x8 db = __builtin_bit_cast(u16x8, d1);
#pragma unroll
        for (int i = 0; i < 8; ++i) S.dz1[unit_of(c, h, i) * kRowStride + at] = db[i];
      }
      const u16x8 xw = __builtin_bit_cast(u16x8, xb);
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (8 * h + i < kIn) S.xs[(8 * h + i) * kRowStride + at] = xw[i];
    }
    wave_sync();
    // dW2 = h1^T dz2 and dW1 = x^T dz1 over the wave's 64 rows; the sums of dz1 and dz2 as products with ones
    // (a thirteenth feature; a tile of its own)
    const auto rows8 = [&](const uint16_t* m, int r, int c) {
      return *reinterpret_cast<const bf16x8_lds*>(m + r * kRowStride + 16 * c + 8 * h);
    };
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      bf16x8 a[2], d[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        a[t] = rows8(S.h1, t * 32 + col, c);
        d[t] = rows8(S.dz2, t * 32 + col, c);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u) dw2[t][u] = mma(a[t], d[u], dw2[t][u]);
      bf16x8 xa = {};
      if (col < kIn) xa = rows8(S.xs, col, c);
      if (col == kIn) xa = ones;
#pragma unroll
      for (int u = 0; u < 2; ++u) dw1[u] = mma(xa, rows8(S.dz1, u * 32 + col, c), dw1[u]);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        db2[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            ones, *reinterpret_cast<const bf16x8_lds*>(S.dz2 + (t * 16 + (l & 15)) * kRowStride + 32 * c + 8 * (l >> 4)),
            db2[t], 0, 0, 0);
    wave_sync();  // the operands are read before the next pass writes them
  }
  for (int off = 16; off > 0; off >>= 1) {
    se += __shfl_xor(se, off);
    db3 += __shfl_xor(db3, off);
  }
  // the wave's partial gradient over its operands' storage, then the block's
  float* P = S.partial;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int j = 0; j < 16; ++j) P[kOffW2 + (t * 32 + acc_row(j)) * kHid + u * 32 + acc_col()] = dw2[t][u][j];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int j = 0; j < 16; ++j)
    {
      const int row = acc_row(j);
      if (row < kIn) P[kOffW1 + row * kHid + u * 32 + acc_col()] = dw1[u][j];
      else if (row == kIn) P[kOffB1 + u * 32 + acc_col()] = dw1[u][j];
    }
  if (l < 16)
#pragma unroll
    for (int t = 0; t < 4; ++t) P[kOffB2 + t * 16 + l] = db2[t][0];
  const int unit = (col >> 4) * 32 + 8 * ((col & 15) >> 2) + 4 * h + (col & 3);  // of value col of this half
  P[kOffW3 + unit] = dw3;
  if (l == 0) P[kOffB3] = db3;
  __shared__ float errors[4];
  if (l == 0) errors[wave] = se;
  __syncthreads();
  for (int i = tid; i < kParams; i += 256)
    partial[static_cast<int64_t>(blockIdx.x) * kParams + i] =
        ((lds[0].partial[i] + lds[1].partial[i]) + lds[2].partial[i]) + lds[3].partial[i];
  if (tid == 0) loss_partial[blockIdx.x] = ((errors[0] + errors[1]) + errors[2]) + errors[3];
}

// The partial gradients summed (sixteen slices of the partials per block of 32 parameters, each in order, then the
// slices in order) and the Adam step.
constexpr int kAdamSlices = 16;
__global__ __launch_bounds__(32 * kAdamSlices) void adam_kernel(const float* partial, int partials, float* grad, float* w,
                                                               float* m, float* v, uint16_t* wb, float lr, float beta1,
                                                               float beta2, float eps, float bc1, float bc2) {
  __shared__ float part[kAdamSlices][32];
  const int slice = threadIdx.x >> 5, i = blockIdx.x * 32 + (threadIdx.x & 31);
  float g = 0.0f;
  if (i < kParams) {
    int k = slice;
    for (; k + 7 * kAdamSlices < partials; k += 8 * kAdamSlices) {  // eight loads ahead of their additions
      float p[8];
      for (int u = 0; u < 8; ++u) p[u] = partial[static_cast<int64_t>(k + u * kAdamSlices) * kParams + i];
      for (int u = 0; u < 8; ++u) g += p[u];
    }
    for (; k < partials; k += kAdamSlices) g += partial[static_cast<int64_t>(k) * kParams + i];
  }
  part[slice][threadIdx.x & 31] = g;
  __syncthreads();
  if (slice != 0 || i >= kParams) return;
  for (int s = 1; s < kAdamSlices; ++s) g += part[s][threadIdx.x];
  grad[i] = g;
  if (lr == 0.0f) return;  // gradients only
  const float mi = beta1 * m[i] + (1.0f - beta1) * g;
  const float vi = beta2 * v[i] + (1.0f - beta2) * g * g;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
  w[i] = wi;
  wb[i] = to_bf16(wi);
}

// A . B (32x8 by 8x32) as the mean of the three matrix instructions that the kernels issue, each with all its k slots
// filled (two and four copies of the eight products) and read back as the kernels read it: an operand or accumulator
// taken from the wrong lane in any of them shows.
__global__ __launch_bounds__(64) void tile_check_kernel(const uint16_t* a, const uint16_t* b, float* c) {
  __shared__ float quarter[32 * 32];
  const int l = threadIdx.x, r = l & 31, h = l >> 5;
  bf16x4 a4, b4;  // the learned sampler's
  bf16x8 a8, b8;  // forward and gradients, k in the order of unit_of
  for (int i = 0; i < 4; ++i) {
    a4[i] = static_cast<short>(a[r * 8 + 4 * h + i]);
    b4[i] = static_cast<short>(b[(4 * h + i) * 32 + r]);
  }
  for (int i = 0; i < 8; ++i) {
    const int k = unit_of(0, h, i) & 7;
    a8[i] = bits_bf16(a[r * 8 + k]);
    b8[i] = bits_bf16(b[k * 32 + r]);
  }
  for (int m0 = 0; m0 < 32; m0 += 16)
    for (int n0 = 0; n0 < 32; n0 += 16) {  // the bias sums'
      bf16x8 at, bt;
      for (int i = 0; i < 8; ++i) {
        at[i] = bits_bf16(a[(m0 + (l & 15)) * 8 + i]);
        bt[i] = bits_bf16(b[i * 32 + n0 + (l & 15)]);
      }
      const f32x4 q = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at, bt, f32x4{}, 0, 0, 0);
      for (int j = 0; j < 4; ++j) quarter[(m0 + 4 * (l >> 4) + j) * 32 + n0 + (l & 15)] = 0.25f * q[j];
    }
  __syncthreads();
  const f32x16 one = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a4, b4, f32x16{}, 0, 0, 0), two = mma(a8, b8, f32x16{});
  for (int j = 0; j < 16; ++j) {
    const int at = acc_row(j) * 32 + acc_col();
    c[at] = (one[j] + 0.5f * two[j] + quarter[at]) / 3.0f;
  }
}

}  // namespace

hipError_t launch_to_bf16(const float* w, uint16_t* wb, int n, hipStream_t stream) {
  to_bf16_kernel<<<(n + 255) / 256, 256, 0, stream>>>(w, wb, n);
  return hipGetLastError();
}

namespace {
bool wide(const float* x) { return (reinterpret_cast<uintptr_t>(x) & 15) == 0; }
}  // namespace

hipError_t launch_forward(const uint16_t* wb, const float* b_fp32, const float* x, int64_t n, float* y,
                          hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  const int64_t blocks = (n + 127) / 128;
  const unsigned grid = static_cast<unsigned>(blocks < 1024 ? blocks : 1024);
  if (wide(x)) forward_kernel<true><<<grid, 256, 0, stream>>>(wb, b_fp32, x, n, y);
  else forward_kernel<false><<<grid, 256, 0, stream>>>(wb, b_fp32, x, n, y);
  return hipGetLastError();
}

int gradient_partials(int64_t n) {
  const int64_t blocks = (n + kStepRows - 1) / kStepRows;
  return static_cast<int>(blocks < kMaxPartials ? blocks : kMaxPartials);
}

hipError_t launch_gradients(const uint16_t* wb, const float* b_fp32, const float* x, const float* target, int64_t n,
                            int64_t batch, float* partial, float* loss_partial, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  const unsigned grid = static_cast<unsigned>(gradient_partials(n));
  const float scale = 2.0f / static_cast<float>(batch);
  if (wide(x)) gradients_kernel<true><<<grid, 256, 0, stream>>>(wb, b_fp32, x, target, n, scale, partial, loss_partial);
  else gradients_kernel<false><<<grid, 256, 0, stream>>>(wb, b_fp32, x, target, n, scale, partial, loss_partial);
  return hipGetLastError();
}

hipError_t launch_adam(const float* partial, int partials, float* grad, float* w, float* m, float* v, uint16_t* wb,
                       const Adam& a, hipStream_t stream) {
  const double bc1 = 1.0 - __builtin_pow(static_cast<double>(a.beta1), a.step);
  const double bc2 = 1.0 - __builtin_pow(static_cast<double>(a.beta2), a.step);
  adam_kernel<<<(kParams + 31) / 32, 32 * kAdamSlices, 0, stream>>>(partial, partials, grad, w, m, v, wb, a.lr, a.beta1, a.beta2,
                                                         a.eps, static_cast<float>(bc1), static_cast<float>(bc2));
  return hipGetLastError();
}

hipError_t launch_tile_check(const uint16_t* a, const uint16_t* b, float* c, hipStream_t stream) {
  tile_check_kernel<<<1, 64, 0, stream>>>(a, b, c);
  return hipGetLastError();
}

}  // namespace mlp
}  // namespace bsx
