// True 32-bit matrix product for the float32 path:  C[n, o] = sum_k A[n, k] * W[o, k], on the matrix cores' bfloat16
// instruction.  A float32 is exactly the sum of three bfloat16 (8 + 8 + 8 bits: high = round(x), middle = round(x - high),
// low = x - high - middle, all differences exact), and a product of two such sums is nine products (the method of Henry, Tang and
// Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for higher-precision computations", 2019), of which the six
// largest are taken, down to high by low at 2^-17 of the whole.  What is left out, middle by low both ways and low by low, is 2^-24 of a product at
// most (a float32 rounding, where the 32-bit instruction has none before its addition) and 2^-27.4 in the root mean square.  Six products at 16 times the
// rate of v_mfma_f32_16x16x4_f32, and 6 additions to a float32 sum for 32 k where that instruction makes 8, which is why a sum's
// error is smaller all the same: relative to the norm, inner size 1,024 2.1e-7 there / 1.6e-7, 4,608 4.3e-7 / 3.7e-7.
//
// The order of a sum.  k is cut into f32_segments(I) stretches of f32_segment(I) values; inside one the sum runs through
// blocks of 32 k in ascending order, the six products of a block smallest first; the stretches' sums are added in ascending
// order.  Both kernels below keep to this whatever tile an element falls in, so a row's result does not depend on how many
// other rows the call holds, and the stretches may be given to different waves.
//
// Values without three such parts.  An infinity or a NaN, and what rounds up to infinity, leaves NaN in its parts, and digits under 2^-133 (of
// values under 2^-110) are lost to bfloat16's smallest value.  What is left of a value behind its second part shows such digits (`collect`:
// half an instruction a value); the rows of A and of W that have any, and the results that are not finite, are taken again on the 32-bit
// matrix instruction from the operands as they are, blocks of 16 x 16 with one such result at a time (`again`).  That depends on a result's own
// two rows alone.  1,194 rows, 9,216 x 1,024 (us, in brackets one lane a result along its rows): none 154, one row with an infinity 250 (664),
// every row with one 892 (6,840); 8 rows of 1,024 x 1,024 5.4, all again 19 (118).
//
// The plain kernel (vector units, ascending k) takes what these refuse: rows that are no whole number of 16 bytes, and
// bfloat16 operands (float32 accumulation) of any size and stride.
#include "f32_parts.h"
#include <algorithm>
#include <utility>

namespace {
// Calls f with the integral constants 0 .. N - 1 (a loop this long the compiler leaves rolled)
template <typename F, int... M>
__device__ __forceinline__ void each(F&& f, std::integer_sequence<int, M...>) { (f(std::integral_constant<int, M>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) { each(f, std::make_integer_sequence<int, N>{}); }

// Tiles of 16 FO WO features x 16 FN WN rows, WO x WN waves of 16 FO x 16 FN.  Both operands are split on their way through registers into
// LDS, in stretches of 32 k; one barrier a stretch.  A part's row of 32 k is 64 bytes, and its 16-byte pieces are exchanged by the
// row, so that the 16 rows of an operand read (16 bytes a lane) lie in 16 different fours of the 64 banks.
// A wave issues in order, and a product keeps the matrix cores busy for 16 cycles, so everything else stands between the products in
// the order written here: the operands' reads a group of products ahead, and the 30 instructions that split and place four values of
// the stretch after the next.  Three stretches in LDS let the reads for the first products of a stretch stand in front of its barrier.
// Workgroup ids go round the 8 chips' L2 caches; the remapping gives each of them whole panels of features, whose rows of W
// then come from memory once.
// SHARED: tiles too few to fill the chip.  The tiles' stretches of k stand in one line, and a workgroup takes `run` of them in a row, so that
// every compute unit gets as much whatever the number of tiles: the end of one tile and the beginning of the next (a run is shorter than
// a tile).  They leave the stretches' sums in `sums` (those from a tile's first on added up) and the rows with lost digits in `marks`, and
// gemm_f32_join_kernel adds the sums in the same order as ever.  1,194 rows, 1,024 features, inner size 4,608: 152 tiles on as many of
// the 256 units 128 us, shared 98; 700 rows 61 (102 in tiles of 32 x 64).
struct SharedSums {
  f32x4* sums;      // [tiles][stretches][FO FN][threads]
  int* marks;       // [tiles][SHARED_PARTS][BO + BN]
  int run;
};
constexpr int SHARED_PARTS = 6;      // workgroups of a tile at most: runs of two and more of at most 8 stretches, and one that they begin within
template <int WO, int WN, int FO, int FN, int OCC, bool SHARED = false>
__global__ __launch_bounds__(64 * WO * WN, OCC) void gemm_f32_tile_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                            float* __restrict__ C, int N, int O, int I, long lda, long ldw,
                                                            long ldc, int row_tiles, int tiles, int wide, SharedSums shared) {
  constexpr int T = 64 * WO * WN, BO = 16 * FO * WO, BN = 16 * FN * WN, ROWS = T / 8, NW = BO / ROWS, NX = BN / ROWS, NP = NW + NX;
  constexpr int PART = (BO + BN) * F32_BK, BUF = 3 * PART;      // a part of both operands (W's rows first), a stretch
  static_assert(NW * ROWS == BO && NX * ROWS == BN && ROWS % 16 == 0, "whole passes, a thread's rows in the same order");
  __shared__ __attribute__((aligned(16))) __bf16 s_p[3 * BUF];
  const int segment = f32_segment(I), stretches = (I + segment - 1) / segment;
  const int groups = SHARED ? (tiles * stretches + shared.run - 1) / shared.run : tiles;
  const int per = (groups + 7) / 8, group = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (group >= groups) return;
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, g = lane / 16, c = lane % 16;
  const int wo = wave / WN * 16 * FO, wn = wave % WN * 16 * FN;
  const int r0 = threadIdx.x / 8, quad = threadIdx.x % 8 * 4;      // this thread's row (of ROWS at a time) and four k of a stretch
  const int at = r0 * F32_BK + ((quad / 8) ^ (r0 / 4 % 4)) * 8 + quad % 8, from = c * F32_BK + (g ^ (c / 4)) * 8;
  // (one tile's stretches from `s_from` on; without SHARED the only one, all of them)
  int line = SHARED ? group * shared.run : group * stretches;
  const int line_end = SHARED ? min(line + shared.run, tiles * stretches) : line + stretches;
  while (true) {
  const int tile = SHARED ? line / stretches : group, s_from = SHARED ? line % stretches : 0;
  const int s_to = SHARED ? min(stretches, s_from + line_end - line) : stretches;
  const int k_from = s_from * segment, k_to = min(s_to * segment, I);
  const int o0 = tile / row_tiles * BO, n0 = tile % row_tiles * BN;
  const float* src[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i)
    src[i] = i < NW ? W + (size_t)min(o0 + r0 + ROWS * i, O - 1) * ldw : A + (size_t)min(n0 + r0 + ROWS * (i - NW), N - 1) * lda;
  f32x4 raw[NP];
  bf16x2 part[3][2];
  uint32_t left[NP] = {};      // (of this thread's rows)
  // (k beyond I: the last four k again, made zero where they are taken up.  No branch may stand there: with one, every wait became a
  // wait for all loads, and the kernel took 1.3 to 1.8 times as long)
  auto ask = [&](int i, int k0) { raw[i] = *(const f32x4*)(src[i] + min(k0 + quad, I - 4)); };
  // a thread's work on four values in eight steps of a few instructions
  constexpr int STEPS = 8;
  auto step = [&](auto index, int buf, int k0, int next) __attribute__((always_inline)) {
    constexpr int i = index.value / STEPS, s = index.value % STEPS;
    f32x4& x = raw[i];
    if constexpr (s == 0 && i >= NW) {      // (of A alone: beyond I both operands hold values of the rows' ends)
      const uint32_t keep = (uint32_t)((k0 + quad - I) >> 31);
      x = __builtin_bit_cast(f32x4, __builtin_bit_cast(u32x4, x) & keep);
    }
    if constexpr (s == 0 || s == 3 || s == 6) {
      part[s / 3][0] = round2(x[0], x[1]);
      part[s / 3][1] = round2(x[2], x[3]);
    }
    if constexpr (s == 1 || s == 4) {
      float x0 = x[0], x1 = x[1];
      take_off(x0, x1, part[s / 3][0]);
      x[0] = x0;
      x[1] = x1;
    }
    if constexpr (s == 2 || s == 5) {
      float x2 = x[2], x3 = x[3];
      take_off(x2, x3, part[s / 3][1]);
      x[2] = x2;
      x[3] = x3;
    }
    if constexpr (s == 6) {
      left[i] = collect(collect(left[i], x[0], x[1]), x[2], x[3]);
      asm("" : "+v"(left[i]));      // (now: put off, it keeps every remainder in a register)
      ask(i, next);
    }
    if constexpr (s == 7) {
#pragma unroll
      for (int q = 0; q < 3; ++q) *(u32x2*)&s_p[buf + q * PART + ROWS * i * F32_BK + at] = u32x2{__builtin_bit_cast(uint32_t, part[q][0]), __builtin_bit_cast(uint32_t, part[q][1])};
    }
  };
  auto read = [&](int buf, int q, int row) { return *(const bf16x8*)&s_p[buf + q * PART + row * F32_BK + from]; };
  f32x4 total[FO][FN] = {};
  bf16x8 fw[3][FO], fx[3][FN], ahead[FN];      // `ahead`: the next stretch's high parts of A
#pragma unroll
  for (int i = 0; i < NP; ++i) ask(i, k_from);
  each<NP * STEPS>([&](auto x) __attribute__((always_inline)) { step(x, 0, k_from, k_from + F32_BK); });
  each<NP * STEPS>([&](auto x) __attribute__((always_inline)) { step(x, BUF, k_from + F32_BK, k_from + 2 * F32_BK); });
  __syncthreads();
#pragma unroll
  for (int i = 0; i < FO; ++i) fw[2][i] = read(0, 2, wo + 16 * i);
#pragma unroll
  for (int i = 0; i < FN; ++i) fx[0][i] = read(0, 0, BO + wn + 16 * i);
  int now = 0, then = BUF, free = 2 * BUF;      // the stretch at hand, the next one, and the one that is filled
  for (int begin = k_from; begin < k_to; begin += segment) {
    const int end = min(begin + segment, I);
    f32x4 acc[FO][FN] = {};
    for (int k0 = begin; k0 < end; k0 += F32_BK) {
      constexpr int G = FO * FN, M = G * F32_PRODUCTS, S = NP * STEPS, R = FO + FN;
      __builtin_amdgcn_sched_barrier(0);
      each<M>([&](auto index) __attribute__((always_inline)) {
        constexpr int m = index.value, p = m / G, t = m % G, i = t / FN, h = t % FN, r0 = t * R / G, s0 = m * S / M;
        acc[i][h] = mfma_bf16(fw[F32_PART[p][0]][i], fx[F32_PART[p][1]][h], acc[i][h]);
        // operands of the products after this group: high W, low A; middle W, A; the next stretch's low W, high A
        if constexpr (p == 0 || p == 1 || p == F32_PRODUCTS - 1)
          each<(t + 1) * R / G - r0>([&](auto j) __attribute__((always_inline)) {
            constexpr int r = r0 + j.value, n = r - FO;
            constexpr int qw = p == 0 ? 0 : (p == 1 ? 1 : 2), qx = p == 0 ? 2 : (p == 1 ? 1 : 0);
            const int buf = p == F32_PRODUCTS - 1 ? then : now;
            if constexpr (r < FO) fw[qw][r] = read(buf, qw, wo + 16 * r);
            else (p == F32_PRODUCTS - 1 ? ahead[n] : fx[qx][n]) = read(buf, qx, BO + wn + 16 * n);
          });
        each<(m + 1) * S / M - s0>([&](auto j) __attribute__((always_inline)) {
          step(std::integral_constant<int, s0 + j.value>{}, free, k0 + 2 * F32_BK, k0 + 3 * F32_BK);
        });
        __builtin_amdgcn_sched_barrier(0);
      });
#pragma unroll
      for (int i = 0; i < FN; ++i) fx[0][i] = ahead[i];
      __syncthreads();
      const int last = now;
      now = then;
      then = free;
      free = last;
    }
#pragma unroll
    for (int i = 0; i < FO; ++i)
#pragma unroll
      for (int h = 0; h < FN; ++h) {
        total[i][h] += acc[i][h];
        if (SHARED && s_from > 0) shared.sums[(((size_t)tile * stretches + begin / segment) * (FO * FN) + i * FN + h) * T + threadIdx.x] = acc[i][h];
      }
  }
  if constexpr (SHARED) {
#pragma unroll
    for (int i = 0; i < FO * FN; ++i)
      if (s_from == 0) shared.sums[(((size_t)tile * stretches + s_to - 1) * (FO * FN) + i) * T + threadIdx.x] = total[i / FN][i % FN];
    int* marks = shared.marks + ((size_t)tile * SHARED_PARTS + group - tile * stretches / shared.run) * (BO + BN);
#pragma unroll
    for (int i = 0; i < NP; ++i) {      // (a row's eight threads are neighbours)
      const uint64_t row = __builtin_amdgcn_ballot_w64(digits_lost(left[i])) >> (lane & ~7) & 0xff;
      if (lane % 8 == 0) marks[ROWS * i + r0] = row != 0;
    }
    line += s_to - s_from;
    if (line >= line_end) return;
    __syncthreads();      // (everyone is done with this tile's operands in LDS)
    continue;
  }
  // which of the tile's rows have lost digits: hardly ever one
  uint32_t any = 0;
#pragma unroll
  for (int i = 0; i < NP; ++i) any |= left[i];
  const bool lost = __syncthreads_or(digits_lost(any));
  int* s_lost = (int*)s_p;      // [BO + BN] (behind the last stretch's barrier, and behind the one above)
  if (__builtin_expect(lost, 0)) {
    for (int i = threadIdx.x; i < BO + BN; i += T) s_lost[i] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (digits_lost(left[i])) s_lost[ROWS * i + r0] = 1;
    __syncthreads();
  }
  static_assert(FO * FN * 4 <= 32, "a bit for each of a lane's results");
  uint32_t want = 0;
#pragma unroll
  for (int i = 0; i < FO; ++i)
#pragma unroll
    for (int h = 0; h < FN; ++h) {
      uint32_t w_lost = 0;
      if (lost) {
#pragma unroll
        for (int j = 0; j < 4; ++j) w_lost |= (uint32_t)s_lost[wo + 16 * i + 4 * g + j] << j;
      }
      want |= wants_again(total[i][h], lost && s_lost[BO + wn + 16 * h + c], w_lost) << (4 * (i * FN + h));
      store_f32x4(C, ldc, n0 + wn + 16 * h + c, o0 + wo + 16 * i + 4 * g, N, O, wide, total[i][h]);
    }
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(want != 0) != 0, 0))
#pragma unroll 1
  for (int b = 0; b < FO * FN; ++b) {
    const uint32_t mine = want >> (4 * b) & 15;
    if (__builtin_amdgcn_ballot_w64(mine != 0) == 0) continue;
    const int row = n0 + wn + 16 * (b % FN) + c, col = o0 + wo + 16 * (b / FN);
    const f32x4 y = again(W + (size_t)min(col + c, O - 1) * ldw, A + (size_t)min(row, N - 1) * lda, I, g, mine);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if ((mine >> j & 1) && row < N && col + 4 * g + j < O) C[(size_t)row * ldc + col + 4 * g + j] = y[j];
  }
  return;
  }
}

// What several workgroups have left of a tile: a block of 16 x 16 a wave has, added in the stretches' order, and the rows that want to be taken again.
template <int WO, int WN, int FO, int FN>
__global__ __launch_bounds__(64 * WO * WN) void gemm_f32_join_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int N,
                                                                     int O, int I, long lda, long ldw, long ldc, int row_tiles, int wide, SharedSums shared) {
  constexpr int T = 64 * WO * WN, BO = 16 * FO * WO, BN = 16 * FN * WN;
  const int segment = f32_segment(I), stretches = (I + segment - 1) / segment;
  const int tile = blockIdx.x, block = blockIdx.y, line = tile * stretches;
  const int first = min(shared.run - line % shared.run, stretches);      // stretches that the first of the tile's workgroups has added up
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, g = lane / 16, c = lane % 16;
  const int wo = wave / WN * 16 * FO + 16 * (block / FN), wn = wave % WN * 16 * FN + 16 * (block % FN);
  const f32x4* sums = shared.sums + ((size_t)line * (FO * FN) + block) * T + threadIdx.x;
  f32x4 sum[F32_SEGMENTS];
#pragma unroll
  for (int s = 0; s < F32_SEGMENTS; ++s) sum[s] = sums[(size_t)min(max(s, first - 1), stretches - 1) * (FO * FN) * T];
  const int parts = (line + stretches - 1) / shared.run - line / shared.run + 1;
  const int* marks = shared.marks + (size_t)tile * SHARED_PARTS * (BO + BN);
  int x_lost = 0;
  uint32_t w_lost = 0;
  for (int p = 0; p < parts; ++p) {
    const int* m = marks + p * (BO + BN);
    x_lost |= m[BO + wn + c];
#pragma unroll
    for (int j = 0; j < 4; ++j) w_lost |= (uint32_t)m[wo + 4 * g + j] << j;
  }
  f32x4 total = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < F32_SEGMENTS; ++s)
    if (s == first - 1) total = sum[s];
    else if (s >= first && s < stretches) total += sum[s];
  const int row = tile % row_tiles * BN + wn + c, col = tile / row_tiles * BO + wo;
  const uint32_t want = wants_again(total, x_lost != 0, w_lost);
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(want != 0) != 0, 0)) {
    const f32x4 y = again(W + (size_t)min(col + c, O - 1) * ldw, A + (size_t)min(row, N - 1) * lda, I, g, want);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (want >> j & 1) total[j] = y[j];
  }
  store_f32x4(C, ldc, row, col + 4 * g, N, O, wide, total);
}

// Few rows or few tiles: a workgroup takes 16 FO features x 16 FN rows and its eight waves a stretch of k each (f32_stretch; no barrier before
// the sums meet in LDS).  Bound by the stream of W (one row group) or by what comes through L2.
template <int FO, int FN>
__global__ __launch_bounds__(512) void gemm_f32_split_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                             float* __restrict__ C, int N, int O, int I, long lda, long ldw,
                                                             long ldc, int wide) {
  __shared__ __attribute__((aligned(16))) f32x4 s_sum[F32_SEGMENTS][FO * FN][WAVE];
  __shared__ __attribute__((aligned(16))) uint64_t s_lost[F32_SEGMENTS];
  const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), g = lane / 16, c = lane % 16;
  const int o0 = blockIdx.x * 16 * FO, n0 = blockIdx.y * 16 * FN;
  const int segments = f32_segments(I), segment = f32_segment(I);
  const int first = wave * segment, last = wave < segments ? min(first + segment, I) : 0;
  const float* wp[FO];
  const float* xp[FN];
#pragma unroll
  for (int i = 0; i < FO; ++i) wp[i] = W + (size_t)min(o0 + 16 * i + c, O - 1) * ldw;
#pragma unroll
  for (int i = 0; i < FN; ++i) xp[i] = A + (size_t)min(n0 + 16 * i + c, N - 1) * lda;
  f32x4 acc[FO][FN] = {};
  uint32_t left[FO + FN] = {};
  f32_stretch(wp, xp, first, last, I, g, acc, left);
  const uint64_t my_lost = rows_lost(left);
  if (lane == 0) s_lost[wave] = my_lost;
#pragma unroll
  for (int i = 0; i < FO; ++i)
#pragma unroll
    for (int h = 0; h < FN; ++h) s_sum[wave][i * FN + h][lane] = acc[i][h];
  __syncthreads();
  uint64_t lost = 0;
#pragma unroll
  for (int s = 0; s < F32_SEGMENTS; ++s) lost |= s_lost[s];
  for (int t = wave; t < FO * FN; t += F32_SEGMENTS) {
    f32x4 total = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < segments; ++s) total += s_sum[s][t][lane];
    const int row = n0 + 16 * (t % FN) + c, col = o0 + 16 * (t / FN);
    total = whole_f32(total, lost, t / FN, FO + t % FN, g, c, I, [&] { return W + (size_t)min(col + c, O - 1) * ldw; }, [&] { return A + (size_t)min(row, N - 1) * lda; });
    store_f32x4(C, ldc, row, col + 4 * g, N, O, wide, total);
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
template <int WO, int WN, int FO, int FN, int OCC>
void launch_tile(const float* A, const float* W, float* C, int N, int O, int I, long lda, long ldw, long ldc, bool wide, hipStream_t stream) {
  const int row_tiles = ceil_div(N, 16 * FN * WN), tiles = row_tiles * ceil_div(O, 16 * FO * WO);
  gemm_f32_tile_kernel<WO, WN, FO, FN, OCC><<<(tiles + 7) / 8 * 8, 64 * WO * WN, 0, stream>>>(A, W, C, N, O, I, lda, ldw, ldc, row_tiles, tiles, wide, SharedSums{});
}
// Tiles of 128 features x 64 rows whose stretches workgroups share: 31 us a tile at an inner size of 1,024 as without, and for the second kernel and the
// sums' way through memory 12 us or, of many tiles, 9 and a sixteenth a tile, whatever the inner size.  (us, without / with, 1,024 features: inner size 4,608
// 150 rows 36.3 / 37.3, 333 69 / 40, 700 102 / 61, 1,194 128 / 98, 1,600 119.1 / 116.5; 4,096 700 rows 92 / 57; 3,072 1,600 rows 82.2 / 84.1; 2,048 1,500 rows
// 58.0 / 55.9, 1,700 59.0 / 64.6; 1,024 333 rows 20.2 / 20.0, 1,194 34.5 / 36.0, 700 rows of 2,048 features 33.4 / 36.9; 4,096 features of inner size 2,048
// 333 rows 61.1 / 58.9, 400 61.5 / 67.4, of 4,096 400 rows 110.7 / 110.9.)
constexpr int SHARED_FEATURES = 128, SHARED_ROWS = 64, SHARED_TILES = 256;
constexpr float SHARED_TILE = 31.f;
struct SharedShape {
  int tiles, stretches, run, groups;
  float cost;      // as the variants' below; 0: does not take the shape
};
SharedShape shared_shape(int N, int O, int I) {
  const int segment = f32_segment(I), stretches = (I + segment - 1) / segment;
  const long tiles = (long)ceil_div(N, SHARED_ROWS) * ceil_div(O, SHARED_FEATURES);
  SharedShape s{(int)tiles, stretches, 0, 0, 0.f};
  if (tiles > SHARED_TILES || I < 2048) return s;      // (256 tiles' sums are 64 MB)
  s.run = std::max(2, (int)ceil_div(tiles * stretches, 256));
  s.groups = ceil_div(tiles * stretches, s.run);
  const float join = fmaxf(12.f, 9.f + tiles / 16.f);
  if (s.run < stretches) s.cost = SHARED_TILE * s.run / stretches + join * 1024.f / I;
  return s;
}
size_t shared_sums_bytes(const SharedShape& s) { return (size_t)s.tiles * s.stretches * SHARED_FEATURES * SHARED_ROWS * 4; }
size_t shared_marks_bytes(const SharedShape& s) { return (size_t)s.tiles * SHARED_PARTS * (SHARED_FEATURES + SHARED_ROWS) * 4; }
void launch_shared(const SharedShape& s, void* work, const float* A, const float* W, float* C, int N, int O, int I, long lda, long ldw, long ldc, bool wide,
                   hipStream_t stream) {
  const SharedSums shared{(f32x4*)work, (int*)((char*)work + shared_sums_bytes(s)), s.run};
  const int row_tiles = ceil_div(N, SHARED_ROWS);
  gemm_f32_tile_kernel<4, 2, 2, 2, 2, true><<<(s.groups + 7) / 8 * 8, 512, 0, stream>>>(A, W, C, N, O, I, lda, ldw, ldc, row_tiles, s.tiles, wide, shared);
  gemm_f32_join_kernel<4, 2, 2, 2><<<dim3(s.tiles, 4), 512, 0, stream>>>(A, W, C, N, O, I, lda, ldw, ldc, row_tiles, wide, shared);
}
template <int FO, int FN>
void launch_split(const float* A, const float* W, float* C, int N, int O, int I, long lda, long ldw, long ldc, bool wide, hipStream_t stream) {
  gemm_f32_split_kernel<FO, FN><<<dim3(ceil_div(O, 16 * FO), ceil_div(N, 16 * FN)), 512, 0, stream>>>(A, W, C, N, O, I, lda, ldw, ldc, wide);
}

// The variants, and which one takes a shape.  A compute unit works through ceil(tiles / 256) tiles; one tile alone takes `alone`, one among
// others on the same unit `loaded` (us at an inner size of 1,024; measured), so the least of max(alone, rounds * loaded) is taken.  Over 1,024
// that order of the variants stays; under it a split tile's waves have four blocks of k or fewer, which are not enough to hide what one
// waits for, and it costs 1.4 times its share.  (77 shapes of 1 to 544 rows and 256 to 6,144 features at 13 inner sizes of 32 to 768, the variant
// taken over the best one, without and with that: in the mean 1.06 and 1.01, at most 2.10 and 1.21; 100 rows x 4,096 features, us:
// inner size 128 10.5 / 6.0, 252 11.9 / 8.6, 512 18.3 / 12.0; inner size 1,024: 1.003, at most 1.05.)
// Features x rows of a tile; the last three cut k over their waves and serve few rows.
// (1,194 rows, us, on the matrix cores' 32-bit instruction / in three parts: 9,216 features x 1,024 227 / 156, 1,024 x 4,608 154 / 123, 1,024 x
// 1,024 38 / 34, 3,072 x 1,024 84 / 50; 333 rows: 9,216 x 1,024 82 / 49; 8 rows: 9,216 x 1,024 11.8 / 12.1, 1,024 x 4,608 15.0 / 15.9, 1,024 x 1,024 5.3 / 5.6
// before the kernels' arguments came in registers, which gives that back: a decoded token of the 350M shape takes as long as it did.)
struct F32Variant {
  int features, rows;
  float alone, loaded;
  void (*launch)(const float*, const float*, float*, int, int, int, long, long, long, bool, hipStream_t);
  bool split;      // k cut over the waves, and rows along the grid's second dimension
};
const F32Variant F32_VARIANTS[] = {
    {128, 128, 41.f, 49.f, launch_tile<2, 4, 4, 2, 2>, false}, {128, 64, 31.f, 34.f, launch_tile<4, 2, 2, 2, 2>, false},
    {64, 64, 26.f, 18.f, launch_tile<2, 2, 2, 2, 2>, false}, {32, 64, 20.f, 13.5f, launch_tile<2, 2, 1, 2, 3>, false},
    {32, 32, 10.f, 9.6f, launch_split<2, 2>, true}, {16, 32, 7.f, 7.f, launch_split<1, 2>, true}, {16, 16, 6.f, 4.2f, launch_split<1, 1>, true}};

// The variant of least cost, which is left in `least`.
const F32Variant* best_variant(int N, int O, int I, float& least) {
  const F32Variant* best = nullptr;
  for (const F32Variant& v : F32_VARIANTS) {
    if (v.split && ceil_div(N, v.rows) > 65535) continue;
    const long tiles = (long)ceil_div(N, v.rows) * ceil_div(O, v.features);
    const float cost = fmaxf(v.alone, (float)((tiles + 255) / 256) * v.loaded) * (v.split && I < 1024 ? 1.4f : 1.f);
    if (!best || cost < least) {
      best = &v;
      least = cost;
    }
  }
  return best;
}
// Whether the stretches are shared where a workspace is there for it.
bool shares(const SharedShape& s, int N, int O, int I) {
  if (s.cost == 0.f) return false;
  float least;
  best_variant(N, O, I, least);
  return s.cost < least;
}
bool launch_f32(const float* A, const float* W, float* C, int N, int O, int I, long lda, long ldw, long ldc, void* work, hipStream_t stream) {
  if (I % 4 || lda % 4 || ldw % 4 || (uintptr_t)A % 16 || (uintptr_t)W % 16) return false;
  const bool wide = O % 4 == 0 && ldc % 4 == 0 && (uintptr_t)C % 16 == 0;
  const SharedShape s = shared_shape(N, O, I);
  float least;
  if (work && shares(s, N, O, I)) launch_shared(s, work, A, W, C, N, O, I, lda, ldw, ldc, wide, stream);
  else best_variant(N, O, I, least)->launch(A, W, C, N, O, I, lda, ldw, ldc, wide, stream);
  return true;
}
}  // namespace

// Bytes of workspace that gibbs_gemm_f32_in can use (0: none; rows that are no whole 16 bytes take the plain kernel).  The results are the same to
// the bit with and without.
GIBBS_EXPORT long gibbs_gemm_f32_workspace(int N, int O, int I) {
  if (N <= 0 || O <= 0 || I <= 0 || I % 4) return 0;
  const SharedShape s = shared_shape(N, O, I);
  return shares(s, N, O, I) ? (long)(shared_sums_bytes(s) + shared_marks_bytes(s)) : 0;
}
// A: [N, I] (row stride lda), W: [O, I] (row stride ldw), C: [N, O] (row stride ldc), all float32; work: null or a workspace of
// gibbs_gemm_f32_workspace bytes, aligned to 16.
GIBBS_EXPORT int gibbs_gemm_f32_in(const float* A, const float* W, float* C, int N, int O, int I, long lda, long ldw, long ldc, void* work,
                                   hipStream_t stream) {
  GIBBS_REQUIRE(N >= 0 && O > 0 && I > 0, "gemm_f32: bad sizes N=%d O=%d I=%d", N, O, I);
  GIBBS_REQUIRE(lda >= I && ldw >= I && ldc >= O, "gemm_f32: row strides shorter than rows");
  GIBBS_REQUIRE((uintptr_t)work % 16 == 0, "gemm_f32: the workspace must be 16-byte aligned");
  if (N == 0) return 0;
  dim3 grid(ceil_div(O, TN), ceil_div(N, TM));
  GIBBS_REQUIRE(grid.y <= 65535, "gemm_f32: too many rows (%d)", N);
  if (launch_f32(A, W, C, N, O, I, lda, ldw, ldc, work, stream)) GIBBS_LAUNCH_STATUS("gemm_f32");
  gemm_plain_kernel<float, float><<<grid, 256, 0, stream>>>(A, W, C, N, O, I, lda, ldw, ldc);
  GIBBS_LAUNCH_STATUS("gemm_f32");
}
GIBBS_EXPORT int gibbs_gemm_f32(const float* A, const float* W, float* C, int N, int O, int I, long lda, long ldw, long ldc, hipStream_t stream) {
  return gibbs_gemm_f32_in(A, W, C, N, O, I, lda, ldw, ldc, nullptr, stream);
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
