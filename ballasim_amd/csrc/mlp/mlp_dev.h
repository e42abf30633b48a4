// Device building blocks of the proposer's kernels: bf16 rounding, the layout of the 32x32 MFMA accumulators, the
// weights in LDS, and the learned sampler's forward pass of one wave's 64 rows (training and inference have their own
// in mlp.hip).
//
// MFMA: v_mfma_f32_32x32x8bf16_1k multiplies a 32x8 bf16 tile A by an 8x32 bf16 tile B into a 32x32
// fp32 accumulator. Lane l (of 64) supplies A[l % 32][4 (l / 32) + i] and B[4 (l / 32) + i][l % 32]
// for i = 0..3, and holds accumulator element j (of 16) at row 8 (j / 4) + 4 (l / 32) + j % 4,
// column l % 32. (launch_tile_check tests the kernels' matrix instructions against a host product.)
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mlp.h"

namespace bsx {
namespace mlp {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

inline constexpr int kS16 = 72;  // row stride (elements) of bf16 LDS matrices: 36 words, no bank aliasing

// fp32 -> bf16, round to nearest even (finite inputs).
__host__ __device__ __forceinline__ uint16_t to_bf16(float f) {
  const uint32_t u = __builtin_bit_cast(uint32_t, f);
  return static_cast<uint16_t>((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}
__host__ __device__ __forceinline__ float from_bf16(uint16_t h) {
  return __builtin_bit_cast(float, static_cast<uint32_t>(h) << 16);
}

// Orders this wave's LDS writes before its lanes read each other's values (the waves of a block run
// their own loops, so no block barrier).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

__device__ __forceinline__ float silu(float z) { return z / (1.0f + __expf(-z)); }

// Row and column of accumulator element j of this lane (row: of the lanes of half h).
__host__ __device__ constexpr int acc_row_of(int j, int h) { return 8 * (j >> 2) + 4 * h + (j & 3); }
__device__ __forceinline__ int acc_row(int j) { return acc_row_of(j, (threadIdx.x & 63) >> 5); }
__device__ __forceinline__ int acc_col() { return threadIdx.x & 31; }

// The weights as the kernels hold them in LDS: bf16 matrices (W1 padded to 16 input rows) and fp32
// biases and output weights (w3 as its bf16 value).
struct WeightsLds {
  uint16_t w1[kInPad * kS16];
  uint16_t w2[kHid * kS16];
  float b1[kHid], b2[kHid], w3[kHid];
  float b3;
};

// ---- One wave's 64 rows (the learned sampler) -------------------------------------------------------
// The products run transposed, hidden units by rows: a lane's accumulators hold 32 units of one row, which,
// rounded to bf16 four at a time, are the next product's B operand as they stand, so activations stay in
// registers. (With the activations and two sets of pre-activations in LDS a wave took 64 KB, which left two waves
// to a compute unit; it takes 15 KB here.) The sums over k and over the output's units run in the order of the
// plain product, so that a sample time does not depend on the layout.
inline constexpr int kS1 = 20, kS2 = 68;  // row strides (elements): 8-byte reads of 32 rows meet every bank once

struct WaveWeights {
  alignas(16) float b1[kHid];
  alignas(16) float b2[kHid];
  float w3[kHid];
  float b3;
  alignas(8) uint16_t w1[kHid * kS1];  // W1 by unit: 16 features (12 and four zeros)
  alignas(8) uint16_t w2[kHid * kS2];  // W2 by output unit
  alignas(8) uint16_t xs[kRowsPerWave * kS1];  // the rows' features, bf16
};

typedef short bf16x4_lds __attribute__((ext_vector_type(4), may_alias));

__device__ __forceinline__ short bf16_bits(float f) { return static_cast<short>(to_bf16(f)); }

// Loads the weights (called by all 64 lanes; lane l takes unit l).
__device__ __forceinline__ void load_weights(WaveWeights& s, const uint16_t* wb, const float* w) {
  const int l = threadIdx.x & 63;
  static_assert(kHid == 64 && kIn % 4 == 0 && kInPad == 16);
#pragma unroll
  for (int q = 0; q < kInPad / 4; ++q) {
    bf16x4 v = {0, 0, 0, 0};
    if (4 * q < kIn)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = static_cast<short>(wb[kOffW1 + (4 * q + i) * kHid + l]);
    *reinterpret_cast<bf16x4_lds*>(s.w1 + l * kS1 + 4 * q) = v;
  }
#pragma unroll
  for (int q = 0; q < kHid / 4; ++q) {
    bf16x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = static_cast<short>(wb[kOffW2 + (4 * q + i) * kHid + l]);
    *reinterpret_cast<bf16x4_lds*>(s.w2 + l * kS2 + 4 * q) = v;
  }
  s.b1[l] = w[kOffB1 + l];
  s.b2[l] = w[kOffB2 + l];
  s.w3[l] = from_bf16(wb[kOffW3 + l]);
  if (l == 0) s.b3 = w[kOffB3];
  wave_sync();
}

// The network's output for each lane's features f[0 .. kIn - 1] (called by all 64 lanes).
__device__ __forceinline__ float wave_forward(WaveWeights& s, const float* f) {
  const int l = threadIdx.x & 63, r = l & 31, kq = (l >> 5) * 4;
#pragma unroll
  for (int q = 0; q < kInPad / 4; ++q) {
    bf16x4 v = {0, 0, 0, 0};
    if (4 * q < kIn)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = bf16_bits(f[4 * q + i]);
    *reinterpret_cast<bf16x4_lds*>(s.xs + l * kS1 + 4 * q) = v;
  }
  wave_sync();
  const auto operand = [](const uint16_t* p) { return *reinterpret_cast<const bf16x4_lds*>(p); };
  uint32_t part[2][32];  // a unit's share of the output of row nt * 32 + l % 32: units acc_row, both tiles
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    bf16x4 h1[8];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      f32x16 acc = {};
#pragma unroll
      for (int k0 = 0; k0 < kInPad; k0 += 8)
        acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(operand(s.w1 + (mt * 32 + r) * kS1 + k0 + kq),
                                                       operand(s.xs + (nt * 32 + r) * kS1 + k0 + kq), acc, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 16; ++j)
        h1[mt * 4 + (j >> 2)][j & 3] = bf16_bits(silu(acc[j] + s.b1[mt * 32 + 8 * (j >> 2) + kq + (j & 3)]));
    }
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      f32x16 acc = {};
#pragma unroll
      for (int k = 0; k < 8; ++k)
        acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(operand(s.w2 + (mt * 32 + r) * kS2 + 8 * k + kq), h1[k], acc,
                                                       0, 0, 0);
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int u = mt * 32 + 8 * (j >> 2) + kq + (j & 3);
        part[nt][mt * 16 + j] = __builtin_bit_cast(uint32_t, from_bf16(to_bf16(silu(acc[j] + s.b2[u]))) * s.w3[u]);
      }
    }
  }
  // Row l is tile l / 32's: the halves exchange what the other's rows need, then each lane adds its row's shares
  // in the order of the units.
  float y = 0.0f;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    float lo[4], hi[4];  // units 8 q + 0 .. 3 and 8 q + 4 .. 7
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const auto both = __builtin_amdgcn_permlane32_swap(part[0][4 * q + i], part[1][4 * q + i], false, false);
      const uint32_t a = both[0], b = both[1];
      lo[i] = __builtin_bit_cast(float, a);
      hi[i] = __builtin_bit_cast(float, b);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) y += lo[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) y += hi[i];
  }
  wave_sync();  // (the next call's features overwrite xs)
  return y + s.b3;
}

}  // namespace mlp
}  // namespace bsx
