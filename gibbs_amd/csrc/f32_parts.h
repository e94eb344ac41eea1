// A float32 product on the matrix cores' bfloat16 instruction: three parts of each operand, six products, the order of the sums, and what is
// taken again in plain float32 (gemm_f32.hip says how and why).  For every kernel whose results must agree with that product to the bit.
#pragma once
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int F32_BK = 32;          // k of a tile in LDS, and of a product
constexpr int F32_SEGMENTS = 8;     // stretches of k with a sum of their own, of 32 k and more
__host__ __device__ inline int f32_segments(int I) { return I >= F32_SEGMENTS * F32_BK ? F32_SEGMENTS : (I + F32_BK - 1) / F32_BK; }
__host__ __device__ inline int f32_segment(int I) {
  const int n = f32_segments(I);
  return ((I + n - 1) / n + F32_BK - 1) / F32_BK * F32_BK;
}

__device__ __forceinline__ f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// Two values to bfloat16 (rounded)
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ bf16x2 round2(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_convertvector((f32x2){a, b}, bf16x2);
}
__device__ __forceinline__ void take_off(float& a, float& b, bf16x2 u) {
  const uint32_t w = __builtin_bit_cast(uint32_t, u);
  a -= __uint_as_float(w << 16);
  b -= __uint_as_float(w & 0xffff0000u);
}
// Eight values x = p[0] + p[1] + p[2], highest first.  What is left of a value is its dot product with (-1, 0) or (0, -1): one
// instruction where take_off has two, and exact like it.  (The tiles' kernel, whose vector instructions stand between products, was
// slower with it.  As constants that the compiler knows, it writes them as -1 for both halves.)
__device__ __forceinline__ void split8(f32x4 x, f32x4 y, bf16x8* p) {
  float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
  uint32_t one = 0xbf80u, two = 0xbf800000u;
  asm volatile("" : "+v"(one), "+v"(two));
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    bf16x2 u[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u[i] = round2(v[2 * i], v[2 * i + 1]);
      if (q < 2) {
        v[2 * i] = __builtin_amdgcn_fdot2_f32_bf16(u[i], __builtin_bit_cast(bf16x2, one), v[2 * i], false);
        v[2 * i + 1] = __builtin_amdgcn_fdot2_f32_bf16(u[i], __builtin_bit_cast(bf16x2, two), v[2 * i + 1], false);
      }
    }
    p[q] = __builtin_shufflevector(__builtin_shufflevector(u[0], u[1], 0, 1, 2, 3), __builtin_shufflevector(u[2], u[3], 0, 1, 2, 3), 0, 1, 2, 3, 4, 5, 6, 7);
  }
}
// The six products of a block, smallest first: (part of the first operand, part of the second)
constexpr int F32_PRODUCTS = 6;
__device__ constexpr int F32_PART[F32_PRODUCTS][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};

__device__ __forceinline__ bool wants_again(float x) { return !(fabsf(x) <= 3.4028234e38f) || (x != 0.f && fabsf(x) < 0x1p-100f); }
// One element in plain float32 (a sum that is NaN stays NaN).
__device__ __forceinline__ float again(const float* a, const float* w, int I) {
  float sum = 0.f;
  for (int k = 0; k < I; k += 4) {
    const f32x4 x = *(const f32x4*)(a + k), y = *(const f32x4*)(w + k);
#pragma unroll
    for (int j = 0; j < 4; ++j) sum = fmaf(x[j], y[j], sum);
    if (sum != sum) break;
  }
  return sum;
}

// Four neighbouring features of one row: lane (g, c) of a product holds features 4 g .. 4 g + 3 of row c.
__device__ __forceinline__ void store_f32x4(float* C, long ldc, int row, int col, int N, int O, bool wide, f32x4 v) {
  if (row >= N || col >= O) return;
  float* p = C + (size_t)row * ldc + col;
  if (wide) {
    *(f32x4*)p = v;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (col + i < O) p[i] = v[i];
  }
}
__device__ __forceinline__ bool wants_again(f32x4 v) { return wants_again(v[0]) || wants_again(v[1]) || wants_again(v[2]) || wants_again(v[3]); }
// The four again, those that want it (few calls ever have one).
__device__ __forceinline__ f32x4 again4(const float* A, const float* W, int I, long lda, long ldw, int row, int col, int N, int O, f32x4 v) {
  if (row < N) {
#pragma unroll 1
    for (int i = 0; i < 4; ++i) {
      const float x = i == 0 ? v[0] : (i == 1 ? v[1] : (i == 2 ? v[2] : v[3]));
      if (col + i >= O || !wants_again(x)) continue;
      const float y = again(A + (size_t)row * lda, W + (size_t)(col + i) * ldw, I);
      v[0] = i == 0 ? y : v[0];
      v[1] = i == 1 ? y : v[1];
      v[2] = i == 2 ? y : v[2];
      v[3] = i == 3 ? y : v[3];
    }
  }
  return v;
}

