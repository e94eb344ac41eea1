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

// One wave's stretch first .. last of a product of 16 FO rows of W with 16 FN of X, straight from memory into the operands' registers, where they are
// split: lane (g, c) reads rows c of wp's and xp's blocks of 16, k 8 g .. 8 g + 7 of a block of 32 (rows of whole 16 bytes, I of them at least 4).
// Four blocks are on their way, and a block is split as soon as it is there (8 rows x 1,024 features, inner size 1,024: 5.6 us; 6.3
// where the first use waited for all loads).
template <int FO, int FN>
__device__ __forceinline__ void f32_stretch(const float* const (&wp)[FO], const float* const (&xp)[FN], int first, int last, int I, int g, f32x4 (&acc)[FO][FN]) {
  constexpr int SETS = 4;
  f32x4 fw[SETS][2][FO], fx[SETS][2][FN];
  // (k beyond the matrix: its last four again, and X's made zero when they are used)
  auto ask = [&](int set, int k0) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int k = min(k0 + 8 * g + 4 * half, I - 4);
#pragma unroll
      for (int i = 0; i < FO; ++i) fw[set][half][i] = *(const f32x4*)(wp[i] + k);
#pragma unroll
      for (int i = 0; i < FN; ++i) fx[set][half][i] = *(const f32x4*)(xp[i] + k);
    }
  };
  auto use = [&](int set, int k0) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const uint32_t keep = (uint32_t)((k0 + 8 * g + 4 * half - I) >> 31);
#pragma unroll
      for (int i = 0; i < FN; ++i) fx[set][half][i] = __builtin_bit_cast(f32x4, __builtin_bit_cast(u32x4, fx[set][half][i]) & keep);
    }
    bf16x8 pw[FO][3], px[FN][3];
#pragma unroll
    for (int i = 0; i < FO; ++i) split8(fw[set][0][i], fw[set][1][i], pw[i]);
#pragma unroll
    for (int i = 0; i < FN; ++i) split8(fx[set][0][i], fx[set][1][i], px[i]);
#pragma unroll
    for (int p = 0; p < F32_PRODUCTS; ++p)
#pragma unroll
      for (int i = 0; i < FO; ++i)
#pragma unroll
        for (int h = 0; h < FN; ++h) acc[i][h] = mfma_bf16(pw[i][F32_PART[p][0]], px[h][F32_PART[p][1]], acc[i][h]);
  };
  // (the first loads stand behind no branch, or the first block's use would wait for all of them: blocks behind a wave's last are that one again)
  if (first < last) {
    const int end = (last - first + 31) / 32 * 32 + first - 32;      // the wave's last block
#pragma unroll
    for (int s = 0; s < SETS; ++s) ask(s, min(first + 32 * s, end));
    int k0 = first;
    for (; k0 + 32 * (2 * SETS - 1) <= end; k0 += 32 * SETS) {
#pragma unroll
      for (int s = 0; s < SETS; ++s) {
        __builtin_amdgcn_sched_barrier(0);
        use(s, k0 + 32 * s);
        ask(s, k0 + 32 * (s + SETS));
      }
    }
#pragma unroll
    for (int s = 0; s < 2 * SETS - 1; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      if (k0 + 32 * s <= end) use(s % SETS, k0 + 32 * s);
      if (s < SETS - 1 && k0 + 32 * (s + SETS) <= end) ask(s, k0 + 32 * (s + SETS));
    }
  }
}

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

