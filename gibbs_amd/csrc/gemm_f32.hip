// True 32-bit matrix product for the float32 path:  C[n, o] = sum_k A[n, k] * W[o, k], on the matrix cores' own 32-bit
// instruction (v_mfma_f32_16x16x4_f32: 32-bit operands, products and sums, 256 flop a cycle and compute unit as on the
// vector units, but without a vector instruction and two LDS reads for every product).
//
// The order of a sum.  k is cut into f32_segments(I) stretches of f32_segment(I) values; inside one the sum runs through
// blocks of 16 k in ascending order, in each of which step j takes the four k that are j modulo 4; the stretches' sums are
// added in ascending order.  Both kernels below keep to this whatever tile an element falls in, so a row's result does not
// depend on how many other rows the call holds, and the stretches may be given to different waves.
//
// The plain kernel (vector units, ascending k) takes what these refuse: rows that are no whole number of 16 bytes, and
// bfloat16 operands (float32 accumulation) of any size and stride.
#include "common.h"

namespace {
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int F32_BK = 32;          // k of a tile in LDS
constexpr int F32_SEGMENTS = 8;     // stretches of k with a sum of their own, for inner sizes of 512 and more
__host__ __device__ inline int f32_segments(int I) { return I >= 512 ? F32_SEGMENTS : 1; }
__host__ __device__ inline int f32_segment(int I) {
  const int n = f32_segments(I);
  return ((I + n - 1) / n + F32_BK - 1) / F32_BK * F32_BK;
}

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

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

// Tiles of 32 FO features x 32 FN rows, four waves of 16 FO x 16 FN; both operands through LDS in stretches of 32 k, the next
// stretch on its way through registers meanwhile, one barrier a stretch.  A row of 32 k lies 36 words apart, so the 16 rows of
// an operand read (16 bytes a lane) start in 16 different fours of the 64 banks.  Bound by the matrix cores: a wave's
// FO x FN x 8 instructions of 32 cycles stand against 2 (FO + FN) reads of LDS.
// Workgroup ids go round the 8 chips' L2 caches; the remapping gives each of them whole panels of features, whose rows of W
// then come from memory once.
template <int FO, int FN>
__global__ __launch_bounds__(256, 2) void gemm_f32_tile_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                            float* __restrict__ C, int N, int O, int I, long lda, long ldw,
                                                            long ldc, int row_tiles, int tiles, int wide) {
  constexpr int BO = 32 * FO, BN = 32 * FN, LD = F32_BK + 4;
  __shared__ __attribute__((aligned(16))) float s_w[2][BO][LD], s_x[2][BN][LD];
  const int per = (tiles + 7) / 8, tile = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (tile >= tiles) return;
  const int o0 = tile / row_tiles * BO, n0 = tile % row_tiles * BN;
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, g = lane / 16, c = lane % 16;
  const int wo = wave / 2 * 16 * FO, wn = wave % 2 * 16 * FN;
  const int r0 = threadIdx.x / 8, quad = threadIdx.x % 8 * 4;      // this thread's row (of 32 at a time) and four k of a stretch
  const float* wp[FO];
  const float* xp[FN];
#pragma unroll
  for (int i = 0; i < FO; ++i) wp[i] = W + (size_t)min(o0 + r0 + 32 * i, O - 1) * ldw + quad;
#pragma unroll
  for (int i = 0; i < FN; ++i) xp[i] = A + (size_t)min(n0 + r0 + 32 * i, N - 1) * lda + quad;
  f32x4 rw[FO], rx[FN];
  // (k beyond I: the last four k again, made zero where the operands are taken up, so that no branch stands between a load
  // and its use; whole stretches of 32 need no such thing, but the one asked for behind the last is that too)
  bool in = true;
  auto ask = [&](int k0) {
    in = k0 + quad < I;
    const int k = in ? k0 : I - 4 - quad;
#pragma unroll
    for (int i = 0; i < FO; ++i) rw[i] = *(const f32x4*)(wp[i] + k);
#pragma unroll
    for (int i = 0; i < FN; ++i) rx[i] = *(const f32x4*)(xp[i] + k);
  };
  auto put = [&](int b) {
#pragma unroll
    for (int i = 0; i < FO; ++i) *(f32x4*)&s_w[b][r0 + 32 * i][quad] = in ? rw[i] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < FN; ++i) *(f32x4*)&s_x[b][r0 + 32 * i][quad] = in ? rx[i] : f32x4{0.f, 0.f, 0.f, 0.f};
  };
  f32x4 total[FO][FN] = {};
  const int segment = f32_segment(I);
  int b = 0;
  ask(0);
  put(0);
  __syncthreads();
  for (int begin = 0; begin < I; begin += segment) {
    const int end = min(begin + segment, I);
    f32x4 acc[FO][FN] = {};
    for (int k0 = begin; k0 < end; k0 += F32_BK, b ^= 1) {
      ask(k0 + F32_BK);
      __builtin_amdgcn_sched_barrier(0);     // (the compiler would move the loads down to where they are used)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        f32x4 fw[FO], fx[FN];
#pragma unroll
        for (int i = 0; i < FO; ++i) fw[i] = *(const f32x4*)&s_w[b][wo + 16 * i + c][16 * half + 4 * g];
#pragma unroll
        for (int i = 0; i < FN; ++i) fx[i] = *(const f32x4*)&s_x[b][wn + 16 * i + c][16 * half + 4 * g];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < FO; ++i)
#pragma unroll
            for (int h = 0; h < FN; ++h) acc[i][h] = mfma_f32(fw[i][j], fx[h][j], acc[i][h]);
      }
      __builtin_amdgcn_sched_barrier(0);     // (nor may what becomes of them be moved up, in front of the products)
      put(b ^ 1);
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < FO; ++i)
#pragma unroll
      for (int h = 0; h < FN; ++h) total[i][h] += acc[i][h];
  }
#pragma unroll
  for (int i = 0; i < FO; ++i)
#pragma unroll
    for (int h = 0; h < FN; ++h) store_f32x4(C, ldc, n0 + wn + 16 * h + c, o0 + wo + 16 * i + 4 * g, N, O, wide, total[i][h]);
}

// Few rows or few tiles: a workgroup takes 16 FO features x 16 FN rows and its eight waves a stretch of k each, straight from
// memory into the operands' registers (no barrier before the sums meet in LDS).  Bound by the stream of W (one row group) or
// by what comes through L2.  The loads of the next 64 k are on their way while the present ones are used.
template <int FO, int FN>
__global__ __launch_bounds__(512) void gemm_f32_split_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                             float* __restrict__ C, int N, int O, int I, long lda, long ldw,
                                                             long ldc, int wide) {
  constexpr int DEEP = 2;           // stretches of 32 k a batch of loads holds
  __shared__ __attribute__((aligned(16))) f32x4 s_sum[F32_SEGMENTS][FO * FN][WAVE];
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, g = lane / 16, c = lane % 16;
  const int o0 = blockIdx.x * 16 * FO, n0 = blockIdx.y * 16 * FN;
  const int segments = f32_segments(I), segment = f32_segment(I);
  const int first = wave * segment, last = wave < segments ? min(first + segment, I) : 0;
  const float* wp[FO];
  const float* xp[FN];
#pragma unroll
  for (int i = 0; i < FO; ++i) wp[i] = W + (size_t)min(o0 + 16 * i + c, O - 1) * ldw;
#pragma unroll
  for (int i = 0; i < FN; ++i) xp[i] = A + (size_t)min(n0 + 16 * i + c, N - 1) * lda;
  f32x4 fw[2][DEEP][2][FO], fx[2][DEEP][2][FN];
  // (k beyond the matrix: its last four again; what lies beyond the wave's stretch is made zero when it is used)
  auto ask = [&](int set, int k0) {
#pragma unroll
    for (int d = 0; d < DEEP; ++d)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int k = min(k0 + 32 * d + 16 * half + 4 * g, I - 4);
#pragma unroll
        for (int i = 0; i < FO; ++i) fw[set][d][half][i] = *(const f32x4*)(wp[i] + k);
#pragma unroll
        for (int i = 0; i < FN; ++i) fx[set][d][half][i] = *(const f32x4*)(xp[i] + k);
      }
  };
  f32x4 acc[FO][FN] = {};
  auto use = [&](int set, int k0) {
    if (k0 + 32 * DEEP > last) {
#pragma unroll
      for (int d = 0; d < DEEP; ++d)
#pragma unroll
        for (int half = 0; half < 2; ++half)
          if (k0 + 32 * d + 16 * half + 4 * g >= last) {
#pragma unroll
            for (int i = 0; i < FO; ++i) fw[set][d][half][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < FN; ++i) fx[set][d][half][i] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
    }
#pragma unroll
    for (int d = 0; d < DEEP; ++d)
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < FO; ++i)
#pragma unroll
            for (int h = 0; h < FN; ++h) acc[i][h] = mfma_f32(fw[set][d][half][i][j], fx[set][d][half][h][j], acc[i][h]);
  };
  if (first < last) {
    ask(0, first);
    for (int k0 = first; k0 < last; k0 += 64 * DEEP) {
      if (k0 + 32 * DEEP < last) ask(1, k0 + 32 * DEEP);
      __builtin_amdgcn_sched_barrier(0);
      use(0, k0);
      if (k0 + 64 * DEEP < last) ask(0, k0 + 64 * DEEP);
      __builtin_amdgcn_sched_barrier(0);
      if (k0 + 32 * DEEP < last) use(1, k0 + 32 * DEEP);
    }
  }
#pragma unroll
  for (int i = 0; i < FO; ++i)
#pragma unroll
    for (int h = 0; h < FN; ++h) s_sum[wave][i * FN + h][lane] = acc[i][h];
  __syncthreads();
  for (int t = wave; t < FO * FN; t += F32_SEGMENTS) {
    f32x4 total = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < segments; ++s) total += s_sum[s][t][lane];
    store_f32x4(C, ldc, n0 + 16 * (t % FN) + c, o0 + 16 * (t / FN) + 4 * g, N, O, wide, total);
  }
}

constexpr int TM = 64, TN = 64, TK = 16;

template <typename T, typename OutT>
__global__ __launch_bounds__(256) void gemm_plain_kernel(const T* __restrict__ A, const T* __restrict__ W,
                                                         OutT* __restrict__ C, int N, int O, int I, long lda,
                                                         long ldw, long ldc) {
  __shared__ float sa[TK][TM + 4];
  __shared__ float sw[TK][TN + 4];
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int row0 = blockIdx.y * TM, col0 = blockIdx.x * TN;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < I; k0 += TK) {
    // 64 rows x 16 k = 1024 elements per operand, 4 per thread.
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = threadIdx.x + i * 256;
      const int r = e / TK, k = e % TK;
      const int gr = row0 + r, gc = col0 + r, gk = k0 + k;
      sa[k][r] = (gr < N && gk < I) ? to_float(A[(size_t)gr * lda + gk]) : 0.f;
      sw[k][r] = (gc < O && gk < I) ? to_float(W[(size_t)gc * ldw + gk]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < TK; ++k) {
      float a[4], w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = sa[k][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = sw[k][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int gr = row0 + ty * 4 + i;
    if (gr >= N) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gc = col0 + tx * 4 + j;
      if (gc < O) C[(size_t)gr * ldc + gc] = from_float<OutT>(acc[i][j]);
    }
  }
}
template <int FO, int FN>
void launch_tile(const float* A, const float* W, float* C, int N, int O, int I, long lda, long ldw, long ldc, bool wide, hipStream_t stream) {
  const int row_tiles = ceil_div(N, 32 * FN), tiles = row_tiles * ceil_div(O, 32 * FO);
  gemm_f32_tile_kernel<FO, FN><<<(tiles + 7) / 8 * 8, 256, 0, stream>>>(A, W, C, N, O, I, lda, ldw, ldc, row_tiles, tiles, wide);
}
template <int FO, int FN>
void launch_split(const float* A, const float* W, float* C, int N, int O, int I, long lda, long ldw, long ldc, bool wide, hipStream_t stream) {
  gemm_f32_split_kernel<FO, FN><<<dim3(ceil_div(O, 16 * FO), ceil_div(N, 16 * FN)), 512, 0, stream>>>(A, W, C, N, O, I, lda, ldw, ldc, wide);
}

// The variants, and which one takes a shape.  A compute unit works through ceil(tiles / 256) tiles; one tile alone takes `alone`, one among
// others on the same unit `loaded` (us at an inner size of 1,024; measured), so the least of max(alone, rounds * loaded) is taken.  Both grow with
// the inner size alike, but for inner sizes under 512, where one wave of a split tile's eight walks all of k: alone it then takes twice
// its share, among others 1.25 times (inner size 508, us, without and with that: 45 rows x 4,096 features 11.0 / 7.5, 300 x 1,024 12.9 / 10.8, 300 x
// 256 7.1 / 5.4).  Features x rows of a tile; the last three cut k over their waves and serve few rows.  (1,194 rows, us, with the vector
// unit's kernel before / now: 9,216 x 1,024 360 / 250, 1,024 x 4,608 640 / 162, 1,024 x 1,024 147 / 39, 3,072 x 1,024 174 / 88;
// 8 rows: 9,216 x 1,024 85 / 15, 1,024 x 4,608 250 / 16.)
struct F32Variant {
  int features, rows;
  float alone, loaded;
  void (*launch)(const float*, const float*, float*, int, int, int, long, long, long, bool, hipStream_t);
  bool split;      // k cut over the waves, and rows along the grid's second dimension
};
const F32Variant F32_VARIANTS[] = {
    {128, 128, 83.f, 78.f, launch_tile<4, 4>, false}, {64, 96, 39.f, 32.f, launch_tile<2, 3>, false}, {64, 64, 28.f, 21.f, launch_tile<2, 2>, false},
    {32, 64, 19.4f, 12.2f, launch_tile<1, 2>, false}, {32, 32, 10.f, 9.6f, launch_split<2, 2>, true}, {16, 32, 6.1f, 6.f, launch_split<1, 2>, true},
    {16, 16, 5.f, 4.2f, launch_split<1, 1>, true}};

bool launch_f32(const float* A, const float* W, float* C, int N, int O, int I, long lda, long ldw, long ldc, hipStream_t stream) {
  if (I % 4 || lda % 4 || ldw % 4 || (uintptr_t)A % 16 || (uintptr_t)W % 16) return false;
  const F32Variant* best = nullptr;
  float least = 0.f;
  for (const F32Variant& v : F32_VARIANTS) {
    if (v.split && ceil_div(N, v.rows) > 65535) continue;
    const long tiles = (long)ceil_div(N, v.rows) * ceil_div(O, v.features);
    const bool one_wave = v.split && f32_segments(I) == 1;
    const float cost = fmaxf(v.alone * (one_wave ? 2.f : 1.f), (float)((tiles + 255) / 256) * v.loaded * (one_wave ? 1.25f : 1.f));
    if (!best || cost < least) {
      best = &v;
      least = cost;
    }
  }
  best->launch(A, W, C, N, O, I, lda, ldw, ldc, O % 4 == 0 && ldc % 4 == 0 && (uintptr_t)C % 16 == 0, stream);
  return true;
}
}  // namespace

// A: [N, I] (row stride lda), W: [O, I] (row stride ldw), C: [N, O] (row stride ldc), all float32.
GIBBS_EXPORT int gibbs_gemm_f32(const float* A, const float* W, float* C, int N, int O, int I, long lda,
                                long ldw, long ldc, hipStream_t stream) {
  GIBBS_REQUIRE(N >= 0 && O > 0 && I > 0, "gemm_f32: bad sizes N=%d O=%d I=%d", N, O, I);
  GIBBS_REQUIRE(lda >= I && ldw >= I && ldc >= O, "gemm_f32: row strides shorter than rows");
  if (N == 0) return 0;
  dim3 grid(ceil_div(O, TN), ceil_div(N, TM));
  GIBBS_REQUIRE(grid.y <= 65535, "gemm_f32: too many rows (%d)", N);
  if (launch_f32(A, W, C, N, O, I, lda, ldw, ldc, stream)) GIBBS_LAUNCH_STATUS("gemm_f32");
  gemm_plain_kernel<float, float><<<grid, 256, 0, stream>>>(A, W, C, N, O, I, lda, ldw, ldc);
  GIBBS_LAUNCH_STATUS("gemm_f32");
}

// A: [N, I], W: [O, I] bfloat16 with any sizes and strides; C: [N, O] bfloat16 (out_dtype 1) or float32 (0).
GIBBS_EXPORT int gibbs_gemm_bf16_plain(const void* A, const void* W, void* C, int out_dtype, int N, int O, int I,
                                       long lda, long ldw, long ldc, hipStream_t stream) {
  GIBBS_REQUIRE(N >= 0 && O > 0 && I > 0, "gemm_bf16_plain: bad sizes N=%d O=%d I=%d", N, O, I);
  GIBBS_REQUIRE(lda >= I && ldw >= I && ldc >= O, "gemm_bf16_plain: row strides shorter than rows");
  if (N == 0) return 0;
  dim3 grid(ceil_div(O, TN), ceil_div(N, TM));
  GIBBS_REQUIRE(grid.y <= 65535, "gemm_bf16_plain: too many rows (%d)", N);
  if (out_dtype == GIBBS_BF16)
    gemm_plain_kernel<bf16, bf16><<<grid, 256, 0, stream>>>((const bf16*)A, (const bf16*)W, (bf16*)C, N, O, I, lda, ldw, ldc);
  else if (out_dtype == GIBBS_F32)
    gemm_plain_kernel<bf16, float><<<grid, 256, 0, stream>>>((const bf16*)A, (const bf16*)W, (float*)C, N, O, I, lda, ldw, ldc);
  else
    return gibbs_fail("gemm_bf16_plain: unknown output dtype %d", out_dtype);
  GIBBS_LAUNCH_STATUS("gemm_bf16_plain");
}
