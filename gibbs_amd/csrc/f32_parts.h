// A float32 product on the matrix cores' bfloat16 instruction: three parts of each operand, six products, the order of the sums, and what is
// taken again on the 32-bit instruction (gemm_f32.hip says how and why).  For every kernel whose results must agree with that product to the bit.
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
// A value that is not the sum of its three parts has digits under 2^-133, bfloat16's smallest value, and 2^-110 is the smallest that can have 24
// bits above it.  What is left of it after two parts shows that: of any other value at most eight bits, whose float32 ends in 16
// zeros.  `left` collects these remainders with OR (one instruction for two values), a row's in one word; whether a row has such a value
// is the row's affair alone, whichever kernel takes it.
__device__ __forceinline__ uint32_t collect(uint32_t left, float a, float b) { return left | __float_as_uint(a) | __float_as_uint(b); }
__device__ __forceinline__ bool digits_lost(uint32_t left) { return (left & 0xffffu) != 0; }
// Eight values x = p[0] + p[1] + p[2], highest first.  What is left of a value is its dot product with (-1, 0) or (0, -1): one
// instruction where take_off has two, and exact like it, subnormal results too.  (The tiles' kernel, whose vector instructions stand between
// products, was slower with it.  As constants that the compiler knows, it writes them as -1 for both halves.)
__device__ __forceinline__ void split8(f32x4 x, f32x4 y, bf16x8* p, uint32_t& left) {
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
      } else {
        left = collect(left, v[2 * i], v[2 * i + 1]);
        asm volatile("" : "+v"(left));      // (now: put off, it keeps every remainder in a register)
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
// `left`: of each of these rows (FO of W, FN of X) what collect gathers of this lane's values.
// Four blocks are on their way, and a block is split as soon as it is there (8 rows x 1,024 features, inner size 1,024: 5.6 us; 6.3
// where the first use waited for all loads).
template <int FO, int FN>
__device__ __forceinline__ void f32_stretch(const float* const (&wp)[FO], const float* const (&xp)[FN], int first, int last, int I, int g, f32x4 (&acc)[FO][FN],
                                            uint32_t (&left)[FO + FN]) {
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
    for (int i = 0; i < FO; ++i) split8(fw[set][0][i], fw[set][1][i], pw[i], left[i]);
#pragma unroll
    for (int i = 0; i < FN; ++i) split8(fx[set][0][i], fx[set][1][i], px[i], left[FO + i]);
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

// Which of the rows have lost digits, 16 bits a block of them (W's blocks first), the same for all lanes of a wave.
template <int BLOCKS>
__device__ __forceinline__ uint64_t rows_lost(const uint32_t (&left)[BLOCKS]) {
  uint64_t rows = 0;
#pragma unroll
  for (int i = 0; i < BLOCKS; ++i) {
    uint64_t m = __builtin_amdgcn_ballot_w64(digits_lost(left[i]));
    m |= m >> 32;
    m |= m >> 16;
    rows |= (m & 0xffff) << (16 * i);
  }
  return rows;
}
// Which of a lane's four results want plain float32: those whose row of X (`x_lost`) or of W (bits of `w_lost`) has lost digits, and those that
// are not finite (an infinity or a NaN leaves NaN in its parts, and so does what rounds up to infinity).
__device__ __forceinline__ uint32_t wants_again(f32x4 v, bool x_lost, uint32_t w_lost) {
  uint32_t want = x_lost ? 15u : w_lost & 15u;
#pragma unroll
  for (int i = 0; i < 4; ++i) want |= (fabsf(v[i]) <= 3.4028234e38f ? 0u : 1u) << i;
  return want;
}
// 16 rows of W by 16 of X in plain float32, on the 32-bit matrix instruction: lane (g, c) has rows c of both (`w`, `x`) and gets
// what mfma_bf16 would give it.  Every lane of the wave takes part.  16 k at a time, four such on their way, until the results that the lanes
// `want` (a bit each) are all NaN.
__device__ __forceinline__ f32x4 again(const float* w, const float* x, int I, int g, uint32_t want) {
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  constexpr int SETS = 4;
#pragma unroll 1
  for (int k0 = 0; k0 < I; k0 += 16 * SETS) {
    f32x4 a[SETS], b[SETS];
#pragma unroll
    for (int s = 0; s < SETS; ++s) {
      const int k = min(k0 + 16 * s + 4 * g, I - 4);
      a[s] = *(const f32x4*)(w + k);
      b[s] = *(const f32x4*)(x + k);
    }
#pragma unroll
    for (int s = 0; s < SETS; ++s) {
      const uint32_t keep = (uint32_t)((k0 + 16 * s + 4 * g - I) >> 31);      // (k beyond I: zero in both)
      const f32x4 p = __builtin_bit_cast(f32x4, __builtin_bit_cast(u32x4, a[s]) & keep), q = __builtin_bit_cast(f32x4, __builtin_bit_cast(u32x4, b[s]) & keep);
#pragma unroll
      for (int j = 0; j < 4; ++j) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(p[j], q[j], sum, 0, 0, 0);
    }
    bool open = false;
#pragma unroll
    for (int j = 0; j < 4; ++j) open |= (want >> j & 1) && sum[j] == sum[j];
    if (__builtin_amdgcn_ballot_w64(open) == 0) break;
  }
  return sum;
}
// The split kernels' results of one block: `lost` says which of the workgroup's rows have lost digits (rows_lost of all waves), wi and xi which of
// its blocks these are; w() and x(): the lane's rows of them.
template <typename WRow, typename XRow>
__device__ __forceinline__ f32x4 whole_f32(f32x4 total, uint64_t lost, int wi, int xi, int g, int c, int I, WRow&& w, XRow&& x) {
  const uint32_t want = wants_again(total, (lost >> (16 * xi + c)) & 1, (uint32_t)(lost >> (16 * wi + 4 * g)));
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(want != 0) != 0, 0)) {
    const f32x4 y = again(w(), x(), I, g, want);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (want >> i & 1) total[i] = y[i];
  }
  return total;
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
