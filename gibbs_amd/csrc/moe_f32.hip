// The experts' products in float32, on the matrix cores in three parts (f32_parts.h): the order of a sum is gemm_f32.hip's and depends on the inner
// size alone, so a pair's result is the same to the bit whatever tile it falls in and whatever else is in the step.
//
// A workgroup takes 16 FN places of one expert's stretch and 32 of its features (gated: 16 of both matrices), its eight waves a stretch of k
// each (f32_stretch); the waves' sums meet in LDS.  Bound by the stream of the experts' matrices for few pairs, by what a compute unit brings
// in for many.
// Width 1,024, experts of 512, 4 of 16 (us, gated and back, vector units before / now): 20 rows 165 and 54 / 18 and 14, 1,000 rows 496
// and 215 / 180 and 145.
#include "activation.h"
#include "f32_parts.h"

namespace {
template <bool GLU, int FN>
__global__ __launch_bounds__(512) void moe_gemm_f32_kernel(const float* __restrict__ X, long ldx, int top, const int* __restrict__ sorted_pair,
                                                           const int* __restrict__ tile_expert, int bm, const float* __restrict__ Wa,
                                                           const float* __restrict__ Wb, long expert_stride, float* __restrict__ Y, long ldy, int O, int I, int act,
                                                           const float* __restrict__ in_weight) {
  constexpr int FO = 2, FEATURES = GLU ? 16 : 32;
  __shared__ __attribute__((aligned(16))) f32x4 s_sum[F32_SEGMENTS][FO * FN][WAVE];
  __shared__ __attribute__((aligned(16))) uint64_t s_lost[F32_SEGMENTS];
  const int p0 = blockIdx.y * 16 * FN, e = tile_expert[p0 / bm];
  if (e < 0 || sorted_pair[p0] < 0) return;      // (an expert's pairs take the first places of its tiles)
  const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), g = lane / 16, c = lane % 16;
  const int o0 = blockIdx.x * FEATURES;
  const int segments = f32_segments(I), segment = f32_segment(I);
  const int first = wave * segment, last = wave < segments ? min(first + segment, I) : 0;
  const float *wa = Wa + (size_t)e * expert_stride, *wb = GLU ? Wb + (size_t)e * expert_stride : wa;
  // (the row of a place without a pair is some row of X, and its results are not stored)
  auto row_of = [&](int place) {
    const int pair = sorted_pair[place];
    return X + (size_t)(pair < 0 ? 0 : (top > 0 ? pair / top : place)) * ldx;
  };
  const float* wp[FO];
  const float* xp[FN];
#pragma unroll
  for (int i = 0; i < FO; ++i) wp[i] = GLU ? (i == 0 ? wa : wb) + (size_t)min(o0 + c, O - 1) * I : wa + (size_t)min(o0 + 16 * i + c, O - 1) * I;
#pragma unroll
  for (int i = 0; i < FN; ++i) xp[i] = row_of(p0 + 16 * i + c);
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
  const bool wide = O % 4 == 0 && ldy % 4 == 0 && ((uintptr_t)Y % 16) == 0;
  uint64_t lost = 0;
#pragma unroll
  for (int s = 0; s < F32_SEGMENTS; ++s) lost |= s_lost[s];
  // the whole sum of one of the workgroup's blocks of results (features from `col` on)
  auto whole = [&](int t, const float* w, int col, const float* x) {
    f32x4 total = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < segments; ++s) total += s_sum[s][t][lane];
    return whole_f32(total, lost, t / FN, FO + t % FN, g, c, I, [&] { return w + (size_t)min(col + c, O - 1) * I; }, [&] { return x; });
  };
  for (int t = wave; t < (GLU ? FN : FO * FN); t += F32_SEGMENTS) {
    const int place = p0 + 16 * (t % FN) + c, pair = sorted_pair[place], col = o0 + 16 * (t / FN);
    const float* x = row_of(place);
    f32x4 v = whole(t, wa, col, x);
    if constexpr (GLU) {
      const f32x4 u = whole(FN + t, wb, col, x);
      const float w = in_weight && pair >= 0 ? in_weight[pair] : 1.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = activate(w * v[i], act) * (w * u[i]);
    }
    if (pair >= 0) store_f32x4(Y, ldy, place, col + 4 * g, place + 1, O, wide, v);
  }
}
}  // namespace

// gibbs_moe_gemm_weighted's float32 products where rows are whole 16 bytes (false: not these operands, nothing was done).
bool moe_gemm_f32(const float* X, long ldx, int top, const int* sorted_pair, const int* tile_expert, long cap, int bm, const float* wa, const float* wb,
                  const float* in_weight, float* Y, long ldy, int O, int I, int act, hipStream_t stream) {
  if (I % 4 || ldx % 4 || (((uintptr_t)X | (uintptr_t)wa | (uintptr_t)wb) % 16)) return false;
  const int fn = bm == 16 ? 1 : 2;      // (places a workgroup takes: many pairs read the matrices half as often)
  const dim3 grid(ceil_div(O, wb ? 16 : 32), (unsigned)(cap / (16 * fn)));
  if (cap / (16 * fn) > 65535) return false;
  auto launch = [&](auto kernel) { kernel<<<grid, 512, 0, stream>>>(X, ldx, top, sorted_pair, tile_expert, bm, wa, wb, (long)O * I, Y, ldy, O, I, act, in_weight); };
  if (wb) fn == 1 ? launch(moe_gemm_f32_kernel<true, 1>) : launch(moe_gemm_f32_kernel<true, 2>);
  else fn == 1 ? launch(moe_gemm_f32_kernel<false, 1>) : launch(moe_gemm_f32_kernel<false, 2>);
  return true;
}
