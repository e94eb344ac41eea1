// Mixture of experts: a router picks `top` of E small gated feed-forwards for every row, and the row's result is
// the weighted sum of theirs; a shared expert may run for every row beside them, times a sigmoid gate of its own.
//
//   route      z = W_r h + b in float32 (h as the step holds it); the `top` largest logits (the lower index among
//              equals); weights = softmax over the chosen logits alone; gate = sigmoid(w_sg . h) for the shared expert
//              (mode 1: scores s = softmax(z) over all router outputs; the `top` largest of s + correction; weights = the
//              chosen scores s divided by their sum + 1e-20, times a constant; mode 2: scores s = sigmoid(z), the `top` largest of s +
//              correction, or of z without one, weights = the chosen scores s as they are.  Router outputs from `E_real` on are identity experts: they
//              have no matrices, their result is the row itself, and their pairs take no place in the tiles)
//   group      the step's (row, choice) pairs sorted by expert into tiles of `bm` pairs that belong to one expert
//              each (every expert's stretch is padded to whole tiles); nothing goes back to the host, so a step
//              with experts can be captured in a graph: the products below run over the worst-case number of tiles
//              and a tile without an expert returns at once
//   gate_up    act[m] = activation(W_gate,e h[row(m)]) * (W_up,e h[row(m)]) for every sorted pair m (rows gathered);
//              with the pairs' weights on their inputs, both products' float32 sums times the pair's weight first
//   down       y[m] = W_down,e act[m]
//   combine    out[row] = sum_c weight[row][c] y[place(row, c)] (ascending c) + gate[row] shared[row], float32 sums
//
// A pair's result depends on nothing but its own row and expert (no sum runs over pairs), so where a pair lands
// among its expert's pairs, which the atomic counters of `group` decide, changes no value: a row's result is the
// same whatever else is in the batch.  Products: plain FMA in ascending k for operands that are not 16-byte aligned; float32 in three bfloat16
// parts on the matrix cores (moe_f32.hip); on the matrix cores for aligned bfloat16, float32 accumulators, the activation in
// float32: tiles of 16 pairs for steps of few pairs (the experts' matrices are streamed once, a workgroup's four
// waves split k, operands straight from memory: rows of h and of every W are contiguous along k), tiles of 128
// pairs beyond (inner sizes of whole tiles of 64 k: 128 pairs x 256 rows of W loaded straight into LDS, three tiles deep, a workgroup a
// compute unit that goes from item to item; others: 128 pairs x 128 or 256 rows of W through registers into LDS in tiles of 32 k,
// double-buffered).
#include "common.h"
#include "activation.h"
#include <algorithm>

// (moe_f32.hip)
bool moe_gemm_f32(const float* X, long ldx, int top, const int* sorted_pair, const int* tile_expert, long cap, int bm, const float* wa, const float* wb,
                  const float* in_weight, float* Y, long ldy, int O, int I, int act, hipStream_t stream);

namespace {
constexpr int MOE_MAX_EXPERTS = 1024;

// ------------------------------------------------------------------------------------------------- route
// 4 neighbouring values of a row as float32 (16-byte or 8-byte loads)
__device__ __forceinline__ float4 load4f(const float* p) { return *(const float4*)p; }
__device__ __forceinline__ float4 load4f(const bf16* p) {
  const uint2 raw = *(const uint2*)p;
  return make_float4(__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u), __uint_as_float(raw.y << 16),
                     __uint_as_float(raw.y & 0xffff0000u));
}
__device__ __forceinline__ void store4f(float* p, float4 v) { *(float4*)p = v; }
__device__ __forceinline__ void store4f(bf16* p, float4 v) {
  union { bf16 h[4]; uint2 u; } o;
  o.h[0] = (bf16)v.x; o.h[1] = (bf16)v.y; o.h[2] = (bf16)v.z; o.h[3] = (bf16)v.w;
  *(uint2*)p = o.u;
}
// One wave's inner products of a row with NV float32 vectors (the row is loaded once); `vec`: the width is a multiple of 4
// and all are aligned, so a lane takes 4 neighbouring values at a time.  Every sum is one chain of additions in ascending
// k per lane, so its value depends on the width alone, not on NV or on how many steps are asked for together.
template <typename T, int NV>
__device__ __forceinline__ void wave_dots(const T* __restrict__ row, const float* const (&w)[NV], float (&out)[NV], int W, int lane, bool vec) {
  float s[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) s[v] = 0.f;
  if (vec) {
    int k = lane * 4;
    // (eight steps at a time, then four: their loads are asked for together)
    for (; k + 7 * WAVE * 4 < W; k += 8 * WAVE * 4) {
      float4 a[8], b[NV][8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        a[u] = load4f(row + k + u * WAVE * 4);
#pragma unroll
        for (int v = 0; v < NV; ++v) b[v][u] = *(const float4*)(w[v] + k + u * WAVE * 4);
      }
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int u = 0; u < 8; ++u) { s[v] = fmaf(a[u].x, b[v][u].x, s[v]); s[v] = fmaf(a[u].y, b[v][u].y, s[v]); s[v] = fmaf(a[u].z, b[v][u].z, s[v]); s[v] = fmaf(a[u].w, b[v][u].w, s[v]); }
    }
    for (; k + 3 * WAVE * 4 < W; k += 4 * WAVE * 4) {
      float4 a[4], b[NV][4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        a[u] = load4f(row + k + u * WAVE * 4);
#pragma unroll
        for (int v = 0; v < NV; ++v) b[v][u] = *(const float4*)(w[v] + k + u * WAVE * 4);
      }
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int u = 0; u < 4; ++u) { s[v] = fmaf(a[u].x, b[v][u].x, s[v]); s[v] = fmaf(a[u].y, b[v][u].y, s[v]); s[v] = fmaf(a[u].z, b[v][u].z, s[v]); s[v] = fmaf(a[u].w, b[v][u].w, s[v]); }
    }
    for (; k < W; k += WAVE * 4) {
      const float4 a = load4f(row + k);
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const float4 c = *(const float4*)(w[v] + k);
        s[v] = fmaf(a.x, c.x, s[v]); s[v] = fmaf(a.y, c.y, s[v]); s[v] = fmaf(a.z, c.z, s[v]); s[v] = fmaf(a.w, c.w, s[v]);
      }
    }
  } else {
    for (int k = lane; k < W; k += WAVE) {
      const float a = to_float(row[k]);
#pragma unroll
      for (int v = 0; v < NV; ++v) s[v] = fmaf(a, w[v][k], s[v]);
    }
  }
#pragma unroll
  for (int v = 0; v < NV; ++v) out[v] = wave_sum(s[v]);
}
template <typename T>
__device__ __forceinline__ float wave_dot(const T* __restrict__ row, const float* __restrict__ w, int W, int lane, bool vec) {
  const float* const ws[1] = {w};
  float out[1];
  wave_dots<T, 1>(row, ws, out, W, lane, vec);
  return out[0];
}

// One wave's choice for row n from its logits z [E] in LDS, which change; `score`: E floats more, for modes 1 and 2.
// the `top` largest, in descending order, the lower index among equal logits (one wave: a lane scans its share of
// the experts, the lanes' bests are folded by exchanges); a logit that was taken becomes NaN; then the softmax
// over the chosen logits alone
__device__ __forceinline__ void choose_experts(float* z, float* score, int n, int lane, const float* __restrict__ router_bias, int* __restrict__ chosen,
                                               float* __restrict__ weight, int E, int top, int mode, float weight_scale, int* __restrict__ place = nullptr,
                                               int matrices = 0) {
  int* mine = chosen + (size_t)n * top;
  float* wts = weight + (size_t)n * top;
  if (mode == 2 && router_bias) {
    for (int e = lane; e < E; e += WAVE) {
      score[e] = 1.0f / (1.0f + expf(-z[e]));
      z[e] = score[e] + router_bias[e];
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
  }
  if (mode == 1) {
    // scores over all outputs; what is compared is the score plus the output's correction
    float zmax = -INFINITY;
    for (int e = lane; e < E; e += WAVE) zmax = fmaxf(zmax, z[e]);
    zmax = wave_max(zmax);
    float total = 0.f;
    for (int e = lane; e < E; e += WAVE) total += expf(z[e] - zmax);
    total = wave_sum(total);
    for (int e = lane; e < E; e += WAVE) {
      const float sc = expf(z[e] - zmax) / total;
      score[e] = sc;
      z[e] = sc + (router_bias ? router_bias[e] : 0.f);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
  }
  // (lane c keeps choice c: a store to memory inside this chain is a wait for it at every turn; 8 rows of 16 experts, 4 chosen, scores over all: 9.3 us so,
  // 8.2 without.  More choices than lanes go to memory as they are made.)
  const bool kept = top <= WAVE;
  int my_pick = -1;
  float my_weight = 0.f, best = 0.f, sum = 0.f;
  for (int c = 0; c < top; ++c) {
    float pv = -INFINITY;
    int pick = 0x7fffffff;
    for (int e = lane; e < E; e += WAVE) {
      const float v = z[e];
      if (v == v && (v > pv || (v == pv && e < pick) || pick == 0x7fffffff)) { pv = v; pick = e; }
    }
    auto meet = [&](float ov, int op) {
      const bool other = op != 0x7fffffff && (pick == 0x7fffffff || ov > pv || (ov == pv && op < pick));
      pv = other ? ov : pv;
      pick = other ? op : pick;
    };
    meet(lane_xor_float<32>(pv), lane_xor_bits<32>(pick));
    meet(lane_xor_float<16>(pv), lane_xor_bits<16>(pick));
    meet(lane_xor_float<8>(pv), lane_xor_bits<8>(pick));
    meet(lane_xor_float<4>(pv), lane_xor_bits<4>(pick));
    meet(lane_xor_float<2>(pv), lane_xor_bits<2>(pick));
    meet(lane_xor_float<1>(pv), lane_xor_bits<1>(pick));
    if (pick == 0x7fffffff) {   // (fewer usable logits than choices: the first expert not taken yet, with no weight)
      __builtin_amdgcn_s_waitcnt(0);
      for (int e = 0; e < E && pick == 0x7fffffff; ++e) {
        bool taken = kept && __builtin_amdgcn_ballot_w64(lane < c && my_pick == e) != 0;
        for (int d = 0; !kept && d < c; ++d) taken |= mine[d] == e;
        if (!taken) pick = e;
      }
      pv = -INFINITY;
    }
    if (c == 0) best = pv;
    const float w = (mode == 1 || (mode == 2 && router_bias)) ? score[pick]
                    : (pv == -INFINITY ? 0.f : (mode == 2 ? 1.0f / (1.0f + expf(-pv)) : expf(pv - best)));
    sum += w;
    if (lane == c) {
      my_pick = pick;
      my_weight = w;
    }
    if (lane == 0) {
      if (!kept) {
        mine[c] = pick;
        wts[c] = w;
      }
      z[pick] = __builtin_nanf("");
    }
    // (the wave's own LDS write above is read by its next scan)
    if (kept) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    else __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
  }
  auto normed = [&](float w) { return mode == 2 ? w : (mode == 1 ? w / (sum + 1e-20f) * weight_scale : (sum > 0.f ? w / sum : 0.f)); };
  if (kept) {
    if (lane < top) {
      mine[lane] = my_pick;
      wts[lane] = normed(my_weight);
      if (place) place[(size_t)n * top + lane] = my_pick < matrices ? n * top + lane : -1;
    }
  } else if (lane == 0) {
    for (int c = 0; c < top; ++c) wts[c] = normed(wts[c]);
  }
}

// The same for at most WAVE experts, a lane each (`correction`: this lane's router_bias, asked for by the caller in front of the logits; 0
// where there is none): a lane counts the experts in front of its own, by descending value and ascending index, NaN behind all, and hands
// its own to the lane of that place.  The same choices, weights and bits: the order is the one in which the turns above take them.  A turn is
// a chain of 0.4 us (LDS, six exchanges, LDS), an expert counted 10 ns: 8 rows of 16 experts, 4 chosen, scores over all, logits included, 8.3 -> 6.7 us;
// 1,992 rows 18.7 -> 16.4.
__device__ __forceinline__ void choose_in_lanes(const float* z, float correction, bool corrected, int n, int lane, int* __restrict__ chosen, float* __restrict__ weight,
                                                int E, int top, int mode, float weight_scale, int* __restrict__ place, int matrices) {
  const bool expert = lane < E;
  float v = expert ? z[lane] : -INFINITY, score = 0.f;
  if (mode == 2 && corrected) {
    score = 1.0f / (1.0f + expf(-v));
    v = score + correction;
  } else if (mode == 1) {
    const float power = expf(v - wave_max(v));
    score = power / wave_sum(expert ? power : 0.f);
    v = score + correction;
  }
  // (whole numbers in the order of the values; both zeros are one number, and NaN lies under -inf)
  const int bits = __float_as_int(v + 0.f), key = v == v ? bits ^ ((bits >> 31) & 0x7fffffff) : (int)0x80000000;
  int ahead = expert ? 0 : lane;
#pragma unroll 8
  for (int e = 0; e < E; ++e) {
    const int other = __builtin_amdgcn_readlane(key, e);
    ahead += expert && other >= key + (e >= lane ? 1 : 0) ? 1 : 0;
  }
  const int pick = __builtin_amdgcn_ds_permute(ahead * 4, lane);
  float pv = __int_as_float(__builtin_amdgcn_ds_permute(ahead * 4, __float_as_int(v)));
  score = __int_as_float(__builtin_amdgcn_ds_permute(ahead * 4, __float_as_int(score)));
  if (!(pv == pv)) pv = -INFINITY;
  const float best = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pv), 0));
  const float w = (mode == 1 || (mode == 2 && corrected)) ? score
                  : (pv == -INFINITY ? 0.f : (mode == 2 ? 1.0f / (1.0f + expf(-pv)) : expf(pv - best)));
  float sum = 0.f;
  for (int c = 0; c < top; ++c) sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), c));
  if (lane < top) {
    chosen[(size_t)n * top + lane] = pick;
    weight[(size_t)n * top + lane] = mode == 2 ? w : (mode == 1 ? w / (sum + 1e-20f) * weight_scale : (sum > 0.f ? w / sum : 0.f));
    if (place) place[(size_t)n * top + lane] = pick < matrices ? n * top + lane : -1;
  }
}

template <typename T>
__global__ __launch_bounds__(1024) void moe_route_kernel(const T* __restrict__ h, long ldh, const float* __restrict__ router,
                                                        const float* __restrict__ router_bias, const float* __restrict__ shared_gate,
                                                        int* __restrict__ chosen, float* __restrict__ weight, float* __restrict__ sgate,
                                                        int W, int E, int top, int mode, float weight_scale, int* __restrict__ place, int matrices) {
  extern __shared__ float z[];   // [E] (mode 1 and 2: and the scores behind them, [E])
  const int n = blockIdx.x, wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, n_waves = blockDim.x / WAVE;
  const T* row = h + (size_t)n * ldh;
  const bool vec = W % 4 == 0 && ldh % 4 == 0 && ((uintptr_t)h % 16) == 0 && ((uintptr_t)router % 16) == 0 && ((uintptr_t)shared_gate % 16) == 0;
  const float correction = router_bias && mode != 0 && wave == 0 && lane < E ? router_bias[lane] : 0.f;
  // the last wave also has the shared expert's gate: with its last expert's logit in one pass over the row
  bool gate_left = shared_gate && wave == n_waves - 1;
  for (int e = wave; e < E; e += n_waves) {
    float s;
    if (gate_left && e + n_waves >= E) {
      const float* const ws[2] = {router + (size_t)e * W, shared_gate};
      float both[2];
      wave_dots<T, 2>(row, ws, both, W, lane, vec);
      s = both[0];
      if (lane == 0) sgate[n] = 1.0f / (1.0f + expf(-both[1]));
      gate_left = false;
    } else {
      s = wave_dot(row, router + (size_t)e * W, W, lane, vec);
    }
    if (lane == 0) z[e] = s + ((router_bias && mode == 0) ? router_bias[e] : 0.f);
  }
  if (gate_left) {
    const float s = wave_dot(row, shared_gate, W, lane, vec);
    if (lane == 0) sgate[n] = 1.0f / (1.0f + expf(-s));
  }
  __syncthreads();
  if (wave != 0) return;
  if (E <= WAVE) choose_in_lanes(z, correction, router_bias != nullptr, n, lane, chosen, weight, E, top, mode, weight_scale, place, matrices);
  else choose_experts(z, z + E, n, lane, router_bias, chosen, weight, E, top, mode, weight_scale, place, matrices);
}

// Many rows: a workgroup of four waves takes four of them, a wave two experts' logits of all four rows at a time, so that a router's row is read
// once for four rows (and a row's values once for two experts), and then a row's choice.  Sums as wave_dots makes them: the same bits.
constexpr int ROUTE_ROWS = 4;
template <typename T>
__global__ __launch_bounds__(ROUTE_ROWS * WAVE) void moe_route_rows_kernel(const T* __restrict__ h, long ldh, const float* __restrict__ router,
                                                                           const float* __restrict__ router_bias, const float* __restrict__ shared_gate,
                                                                           int* __restrict__ chosen, float* __restrict__ weight, float* __restrict__ sgate, int N,
                                                                           int W, int E, int top, int mode, float weight_scale) {
  extern __shared__ float z[];   // [ROUTE_ROWS][E], and as many scores behind them
  const int n0 = blockIdx.x * ROUTE_ROWS, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  const int vectors = E + (shared_gate ? 1 : 0);
  const float correction = router_bias && mode != 0 && lane < E ? router_bias[lane] : 0.f;
  const T* rows[ROUTE_ROWS];
#pragma unroll
  for (int r = 0; r < ROUTE_ROWS; ++r) rows[r] = h + (size_t)min(n0 + r, N - 1) * ldh;
  for (int e = 2 * wave; e < vectors; e += 2 * ROUTE_ROWS) {
    const float* w[2];
#pragma unroll
    for (int v = 0; v < 2; ++v) w[v] = min(e + v, vectors - 1) < E ? router + (size_t)min(e + v, vectors - 1) * W : shared_gate;
    float s[2][ROUTE_ROWS] = {};
    auto step = [&](const float4 (&a)[ROUTE_ROWS], const float4 (&b)[2]) {
#pragma unroll
      for (int v = 0; v < 2; ++v)
#pragma unroll
        for (int r = 0; r < ROUTE_ROWS; ++r) {
          s[v][r] = fmaf(a[r].x, b[v].x, s[v][r]); s[v][r] = fmaf(a[r].y, b[v].y, s[v][r]);
          s[v][r] = fmaf(a[r].z, b[v].z, s[v][r]); s[v][r] = fmaf(a[r].w, b[v].w, s[v][r]);
        }
    };
    int k = lane * 4;
    for (; k + WAVE * 4 < W; k += 2 * WAVE * 4) {
      float4 a[2][ROUTE_ROWS], b[2][2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int r = 0; r < ROUTE_ROWS; ++r) a[u][r] = load4f(rows[r] + k + u * WAVE * 4);
#pragma unroll
        for (int v = 0; v < 2; ++v) b[u][v] = *(const float4*)(w[v] + k + u * WAVE * 4);
      }
      step(a[0], b[0]);
      step(a[1], b[1]);
    }
    for (; k < W; k += WAVE * 4) {
      float4 a[ROUTE_ROWS], b[2];
#pragma unroll
      for (int r = 0; r < ROUTE_ROWS; ++r) a[r] = load4f(rows[r] + k);
#pragma unroll
      for (int v = 0; v < 2; ++v) b[v] = *(const float4*)(w[v] + k);
      step(a, b);
    }
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int r = 0; r < ROUTE_ROWS; ++r) {
        const float sum = wave_sum(s[v][r]);
        if (lane != 0 || e + v >= vectors) continue;
        if (e + v < E) z[r * E + e + v] = sum + ((router_bias && mode == 0) ? router_bias[e + v] : 0.f);
        else if (n0 + r < N) sgate[n0 + r] = 1.0f / (1.0f + expf(-sum));
      }
  }
  __syncthreads();
  if (n0 + wave >= N) return;
  if (E <= WAVE) choose_in_lanes(z + wave * E, correction, router_bias != nullptr, n0 + wave, lane, chosen, weight, E, top, mode, weight_scale, nullptr, 0);
  else choose_experts(z + wave * E, z + (ROUTE_ROWS + wave) * E, n0 + wave, lane, router_bias, chosen, weight, E, top, mode, weight_scale);
}

// ------------------------------------------------------------------------------------------------- group
// One workgroup: counts per expert, every expert's stretch rounded up to whole tiles, then each pair takes the next
// free place of its expert's stretch.  sorted_pair [cap]: the pair at each place (-1: padding); pair_pos [n_pairs]:
// each pair's place; tile_expert [cap / bm]: the expert of each tile (-1: beyond the last stretch).
// (a pair whose expert is E or beyond, an identity expert, gets the place -1)
__global__ __launch_bounds__(1024) void moe_group_kernel(const int* __restrict__ chosen, int n_pairs, int E, int bm,
                                                         int* __restrict__ sorted_pair, int* __restrict__ pair_pos,
                                                         int* __restrict__ tile_expert, int cap) {
  __shared__ int count[MOE_MAX_EXPERTS];
  __shared__ int start[MOE_MAX_EXPERTS + 1];
  for (int e = threadIdx.x; e < E; e += blockDim.x) count[e] = 0;
  for (int m = threadIdx.x; m < cap; m += blockDim.x) sorted_pair[m] = -1;
  __syncthreads();
  for (int i = threadIdx.x; i < n_pairs; i += blockDim.x)
    if (chosen[i] < E) atomicAdd(&count[chosen[i]], 1);
  __syncthreads();
  if (threadIdx.x == 0) {
    int at = 0;
    for (int e = 0; e < E; ++e) {
      start[e] = at;
      at += (count[e] + bm - 1) / bm * bm;
    }
    start[E] = at;
  }
  __syncthreads();
  for (int t = threadIdx.x; t < cap / bm; t += blockDim.x) {
    const int m = t * bm;
    int e = -1;
    if (m < start[E]) {   // the expert whose stretch holds place m
      int lo = 0, hi = E - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (start[mid] <= m) lo = mid; else hi = mid - 1;
      }
      e = lo;
    }
    tile_expert[t] = e;
  }
  for (int e = threadIdx.x; e < E; e += blockDim.x) count[e] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < n_pairs; i += blockDim.x) {
    const int e = chosen[i];
    if (e >= E) { pair_pos[i] = -1; continue; }
    const int m = start[e] + atomicAdd(&count[e], 1);
    sorted_pair[m] = i;
    pair_pos[i] = m;
  }
}

// ------------------------------------------------------------------------------------------------- products, plain
// Tile of BM places x 64 features; thread (feature tx, row lane ty of 4) keeps BM / 4 rows of its feature; every sum
// in ascending k.  GLU: two matrices and act(gate) * up; else one matrix.  X rows: gathered by pair (pair / top) when
// `top` > 0, else the places themselves.
template <typename T, int BM, bool GLU>
__global__ __launch_bounds__(256) void moe_gemm_plain_kernel(const T* __restrict__ X, long ldx, int top, const int* __restrict__ sorted_pair,
                                                             const int* __restrict__ tile_expert, const T* __restrict__ Wa,
                                                             const T* __restrict__ Wb, long expert_stride, T* __restrict__ Y, long ldy,
                                                             int O, int I, int act, const float* __restrict__ in_weight) {
  constexpr int TK = 16, RPT = BM / 4;
  __shared__ float sx[TK][BM + 1];
  __shared__ float sa[TK][64 + 1];
  __shared__ float sb[GLU ? TK : 1][64 + 1];
  __shared__ int src[BM];
  const int tile = blockIdx.y, e = tile_expert[tile];
  if (e < 0) return;
  const int col0 = blockIdx.x * 64, tx = threadIdx.x % 64, ty = threadIdx.x / 64;
  if (threadIdx.x < BM) {
    const int pair = sorted_pair[tile * BM + threadIdx.x];
    src[threadIdx.x] = pair < 0 ? -1 : (top > 0 ? pair / top : tile * BM + threadIdx.x);
  }
  __syncthreads();
  const T* wa = Wa + (size_t)e * expert_stride;
  const T* wb = GLU ? Wb + (size_t)e * expert_stride : nullptr;
  float acc_a[RPT] = {}, acc_b[RPT] = {};
  for (int k0 = 0; k0 < I; k0 += TK) {
    for (int i = threadIdx.x; i < TK * BM; i += 256) {
      const int r = i / TK, k = i % TK;
      sx[k][r] = (src[r] >= 0 && k0 + k < I) ? to_float(X[(size_t)src[r] * ldx + k0 + k]) : 0.f;
    }
    for (int i = threadIdx.x; i < TK * 64; i += 256) {
      const int c = i / TK, k = i % TK;
      const bool in = col0 + c < O && k0 + k < I;
      sa[k][c] = in ? to_float(wa[(size_t)(col0 + c) * I + k0 + k]) : 0.f;
      if (GLU) sb[k][c] = in ? to_float(wb[(size_t)(col0 + c) * I + k0 + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < TK; ++k) {
      const float a = sa[k][tx], b = GLU ? sb[k][tx] : 0.f;
#pragma unroll
      for (int r = 0; r < RPT; ++r) {
        const float x = sx[k][ty + 4 * r];
        acc_a[r] = fmaf(x, a, acc_a[r]);
        if (GLU) acc_b[r] = fmaf(x, b, acc_b[r]);
      }
    }
    __syncthreads();
  }
  if (col0 + tx >= O) return;
#pragma unroll
  for (int r = 0; r < RPT; ++r) {
    const int row = ty + 4 * r;
    if (src[row] < 0) continue;
    const float w = (GLU && in_weight) ? in_weight[sorted_pair[tile * BM + row]] : 1.f;
    const float v = GLU ? activate(w * acc_a[r], act) * (w * acc_b[r]) : acc_a[r];
    Y[(size_t)(tile * BM + row) * ldy + col0 + tx] = from_float<T>(v);
  }
}

// ------------------------------------------------------------------------------------------------- products, matrix cores
// bfloat16, inner size a multiple of 8, rows 16-byte aligned.
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

// Few pairs: a tile is 16 places, a workgroup takes 16 NF features of it (GLU: of both matrices) and its four waves a
// quarter of k each, so that the experts' matrices, which are read once, are spread over many workgroups; the waves'
// sums meet in LDS and are added in wave order.  W is the first operand of the 16 x 16 x 32 product (the
// tile is Y^T = W X^T): lane l holds 8 values along k of feature or place l % 16, and its four results are four
// neighbouring features of place l % 16.  Operands come straight from memory.  Measured (16 experts of 1,024 at width 2,048, 4 chosen; us, gated and
// back): 1 row 13.7 and 6.7 with loads under conditions, 32 features and one wave's tail, 10.1 and 5.6 now; 8 rows (126 and 63 MB) 34.8 and
// 13.7, now 27.0 and 12.9; back with 16 features a workgroup or 32, 8 rows 13.7 / 13.1 (gated: gibbs_moe_gated_features).
// DIRECT (at most 64 pairs, an expert at most 16 of them): no grouping in front: `sorted_pair` holds each pair's choice, places are the pairs' own
// numbers, and the workgroups are laid out over the experts that are chosen, not over all: with a grid of all of them the chosen ones' could meet on
// the same compute units (16 experts, 2 rows, 7 of them chosen: gated 20.4 us and back 11.8, now 12.7 and 8.2).  Finding its expert costs a workgroup 0.1 to 0.2
// us, which one row's products back feel (5.6 -> 5.8 us).
// TURN: workgroups begin at different k (few_turns).
template <bool GLU, bool DIRECT, int NF, bool TURN>
__global__ __launch_bounds__(256) void moe_gemm_few_kernel(const bf16* __restrict__ X, const int* __restrict__ sorted_pair,
                                                           const int* __restrict__ tile_expert, const bf16* __restrict__ Wa,
                                                           const bf16* __restrict__ Wb, int top, int I, long ldx, long expert_stride, bf16* __restrict__ Y,
                                                           long ldy, int O, int act, const float* __restrict__ in_weight, int pairs, int experts) {
  constexpr int NA = GLU ? 2 * NF : NF;    // accumulators a wave
  __shared__ __attribute__((aligned(16))) floatx4 part[4][NA][WAVE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE, lr = lane % 16, lg = lane / 16;
  int e, pair, place;
  if constexpr (DIRECT) {
    const int choice = sorted_pair[min(lane, pairs - 1)];
    // the pairs with a lane's own choice, by the choices' bits; the `nth` expert of those chosen is the one whose first pair is the nth such
    const bool live = lane < pairs && (unsigned)choice < (unsigned)experts;
    uint64_t same = __builtin_amdgcn_ballot_w64(live);
    for (int b = 0; (experts - 1) >> b; b += 4)      // (bits that no choice has change nothing)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const bool bit = choice >> (b + u) & 1;
        const uint64_t with = __builtin_amdgcn_ballot_w64(bit);
        same &= bit ? with : ~with;
      }
    const bool first = live && __builtin_ctzll(same) == lane;
    const uint64_t firsts = __builtin_amdgcn_ballot_w64(first), found = __builtin_amdgcn_ballot_w64(first && __popcll(firsts & ((1ull << lane) - 1)) == (int)blockIdx.y);
    if (found == 0) return;
    e = __builtin_amdgcn_readlane(choice, __builtin_ctzll(found));
    const uint64_t all = __builtin_amdgcn_ballot_w64(live && choice == e);
    // the expert's pairs, in ascending order, to lanes 0, 1, ...; every lane then takes its place's
    const int rank = __popcll(all & ((1ull << lane) - 1));
    const int sent = __builtin_amdgcn_ds_permute((all >> lane & 1 ? rank : WAVE - 1) * 4, lane);
    pair = __builtin_amdgcn_ds_bpermute(lr * 4, sent);
    if (lr >= __popcll(all)) pair = -1;
    place = pair < 0 ? 0 : pair;
  } else {
    e = tile_expert[blockIdx.y];
    place = blockIdx.y * 16 + lr;
    pair = sorted_pair[place];
    if (e < 0) return;
  }
  const int col0 = blockIdx.x * (16 * NF);
  const int src = pair < 0 ? 0 : (top > 0 ? pair / top : place);      // (a place without a pair: some row, its results are not stored)
  const bf16* xr = X + (size_t)src * ldx;
  const bf16* w[NA];
#pragma unroll
  for (int t = 0; t < NA; ++t) w[t] = (GLU && t >= NF ? Wb : Wa) + (size_t)e * expert_stride + (size_t)min(col0 + t % NF * 16 + lr, O - 1) * I;
  floatx4 acc[NA];
#pragma unroll
  for (int t = 0; t < NA; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  // wave w takes the stretches of 64 along k whose number is w modulo 4, in ascending order.  A lane group holds 16
  // neighbouring values of a stretch as the operands of two products (the order along k inside a product is free as long as
  // both operands agree), so that the wave asks for whole lines of 128 bytes of every row; two stretches on their way.  No load stands
  // under a condition (each would be waited for alone): k beyond I reads the rows' last values, and X's are made zero.
  const int n = I > wave * 64 ? (I - wave * 64 + 255) / 256 : 0;      // this wave's stretches
  bf16x8 x8[2][2], w8[2][2][NA];
  auto ask = [&](int set, int it) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint32_t k = min(it * 256 + wave * 64 + lg * 16 + u * 8, I - 8);
      x8[set][u] = *(const bf16x8*)(xr + k);
#pragma unroll
      for (int t = 0; t < NA; ++t) w8[set][u][t] = *(const bf16x8*)(w[t] + k);
    }
  };
  auto use = [&](int set, int it) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (it * 256 + wave * 64 + 64 > I && it * 256 + wave * 64 + lg * 16 + u * 8 >= I) x8[set][u] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int t = 0; t < NA; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w8[set][u][t], x8[set][u], acc[t], 0, 0, 0);
    }
  };
  if (n > 0) {
    // The workgroups begin at different k: rows of 4 KB and more, all read at one k at a time, are a few of the memory's channels (8 and 32 rows, gated,
    // 32.1 and 35.5 us without, 27.0 and 30.4; rows of 2 KB, back, 13.1 / 13.4).  By the feature, so that a result's sum does not depend on the grid.
    const int turn = TURN ? col0 / 32 % n : 0;
    auto nth = [&](int it) { return !TURN || it + turn < n ? it + turn : it + turn - n; };
    ask(0, nth(0));
    ask(1, nth(min(1, n - 1)));
    int it = 0;
    for (; it + 2 < n; it += 2) {
      use(0, nth(it));
      ask(0, nth(it + 2));
      __builtin_amdgcn_sched_barrier(0x7 | 0x8 | 0x380);
      use(1, nth(it + 1));
      ask(1, nth(min(it + 3, n - 1)));
      __builtin_amdgcn_sched_barrier(0x7 | 0x8 | 0x380);
    }
    use(0, nth(it));
    if (it + 1 < n) use(1, nth(it + 1));
  }
#pragma unroll
  for (int t = 0; t < NA; ++t) part[wave][t][lane] = acc[t];
  __syncthreads();
  if (wave >= NF || pair < 0) return;      // wave t writes features t * 16 .. + 16
  const float pw = (GLU && in_weight) ? in_weight[pair] : 1.f;
  floatx4 pa[4], pb[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    pa[v] = part[v][wave][lane];
    if (GLU) pb[v] = part[v][GLU ? NF + wave : 0][lane];
  }
  floatx4 a = {0.f, 0.f, 0.f, 0.f}, b = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    a += pa[v];
    if (GLU) b += pb[v];
  }
  if (GLU) {
    // (which activation is asked once, not for each value)
    a *= pw;
    if (act == ACT_SILU) {
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = activate(a[i], ACT_SILU) * (pw * b[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = activate(a[i], act) * (pw * b[i]);
    }
  }
  const int col = col0 + wave * 16 + lg * 4;
  bf16* y = Y + (size_t)place * ldy + col;
  if (col + 3 < O && ldy % 4 == 0 && ((uintptr_t)Y % 8) == 0) {
    *(bf16x4*)y = bf16x4{(bf16)a[0], (bf16)a[1], (bf16)a[2], (bf16)a[3]};
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (col + i < O) y[i] = (bf16)a[i];
  }
}

// Many pairs: a tile is 128 places, a workgroup of NW waves computes 128 places x BN rows of W (GLU: BN / 2 features of both
// matrices), each wave 64 x 64 as 2 x 2 products of 32 x 32 x 16; tiles of BK along k go through LDS (rows padded by 16
// bytes against bank conflicts), double-buffered, and a further tile waits in registers, so that a tile's loads have
// two tiles' work to arrive.  The rows of X are gathered by the tile's pairs as they are loaded.
constexpr int TBM = 128;
template <int BK, int BN>
struct MoeTile {
  bf16 a[TBM][BK + 8];
  bf16 w[BN][BK + 8];
};
template <bool GLU, int BK, int BN, int NW>
__global__ __launch_bounds__(NW * WAVE) void moe_gemm_tiled_kernel(const bf16* __restrict__ X, long ldx, int top, const int* __restrict__ sorted_pair,
                                                             const int* __restrict__ tile_expert, const bf16* __restrict__ Wa,
                                                             const bf16* __restrict__ Wb, long expert_stride, bf16* __restrict__ Y, long ldy,
                                                             int O, int I, int act, const float* __restrict__ in_weight) {
  using Tile = MoeTile<BK, BN>;
  constexpr int KC = BK / 8;                        // chunks of 16 bytes in a row of a tile
  constexpr int THREADS = NW * WAVE, WN = NW / 2;   // waves: 2 along the places, WN along the rows of W
  constexpr int CA = TBM * KC / THREADS, CW = BN * KC / THREADS;   // chunks a thread moves per operand and tile of k
  constexpr int NT = BN / WN / 32;                  // column blocks of 32 a wave
  static_assert(CA >= 1 && CW >= 1 && NT >= (GLU ? 2 : 1) && NT % (GLU ? 2 : 1) == 0, "tile sizes");
  extern __shared__ __attribute__((aligned(16))) char moe_lds[];
  Tile* tiles = (Tile*)moe_lds;                     // [2]
  int* srcs = (int*)(moe_lds + 2 * sizeof(Tile));   // [TBM]
  float* pair_w = (float*)(srcs + TBM);             // [TBM]: the pairs' weights on their inputs (1 without)
  const int tile = blockIdx.y, e = tile_expert[tile];
  if (e < 0) return;
  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
  constexpr int COLS = GLU ? BN / 2 : BN;           // features of the result that a workgroup takes
  const int col0 = blockIdx.x * COLS;
  if (tid < TBM) {
    const int pair = sorted_pair[tile * TBM + tid];
    srcs[tid] = pair < 0 ? -1 : (top > 0 ? pair / top : tile * TBM + tid);
    if (GLU) pair_w[tid] = (in_weight && pair >= 0) ? in_weight[pair] : 1.f;
  }
  __syncthreads();
  const bf16* wa = Wa + (size_t)e * expert_stride;
  const bf16* wb = GLU ? Wb + (size_t)e * expert_stride : nullptr;
  const int wr = (wave / WN) * 64;
  // a thread's rows stay the same from tile to tile
  const bf16* pa[CA];
  const bf16* pw[CW];
#pragma unroll
  for (int i = 0; i < CA; ++i) {
    const int r = (tid + i * THREADS) / KC;
    pa[i] = srcs[r] >= 0 ? X + (size_t)srcs[r] * ldx : nullptr;
  }
#pragma unroll
  for (int i = 0; i < CW; ++i) {
    const int r = (tid + i * THREADS) / KC;
    const int col = col0 + (GLU ? r % COLS : r);
    pw[i] = col < O ? ((GLU && r >= COLS) ? wb : wa) + (size_t)col * I : nullptr;
  }
  // two register sets take turns: a tile's loads are asked for two tiles ahead of its use
  uint4 ra[2][CA], rw[2][CW];
  auto load_global = [&](int k0, uint4* a, uint4* w) {
    const int gk = k0 + (tid % KC) * 8;
#pragma unroll
    for (int i = 0; i < CA; ++i) a[i] = (pa[i] && gk < I) ? *(const uint4*)(pa[i] + gk) : make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < CW; ++i) w[i] = (pw[i] && gk < I) ? *(const uint4*)(pw[i] + gk) : make_uint4(0, 0, 0, 0);
  };
  auto store_lds = [&](Tile& t, const uint4* a, const uint4* w) {
    const int kc = (tid % KC) * 8;
#pragma unroll
    for (int i = 0; i < CA; ++i) *(uint4*)&t.a[(tid + i * THREADS) / KC][kc] = a[i];
#pragma unroll
    for (int i = 0; i < CW; ++i) *(uint4*)&t.w[(tid + i * THREADS) / KC][kc] = w[i];
  };
  floatx16 acc[2][NT];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[m][n][i] = 0.f;
  // the wave's column blocks of 32 in the W tile: neighbours (one matrix), or the same features of gate (the first half of
  // its blocks) and up (the second half)
  int wc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
    wc[n] = GLU ? (n / (NT / 2)) * COLS + (wave % WN) * (COLS / WN) + (n % (NT / 2)) * 32 : (wave % WN) * (BN / WN) + n * 32;
  const int n_tiles = (I + BK - 1) / BK;
  auto compute = [&](const Tile& cur) {
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      bf16x8 fa[2], fw[NT];
      const int k = kk * 16 + (lane / 32) * 8;
#pragma unroll
      for (int m = 0; m < 2; ++m) fa[m] = *(const bf16x8*)&cur.a[wr + m * 32 + lane % 32][k];
#pragma unroll
      for (int n = 0; n < NT; ++n) fw[n] = *(const bf16x8*)&cur.w[wc[n] + lane % 32][k];
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[m], fw[n], acc[m][n], 0, 0, 0);
    }
  };
  load_global(0, ra[0], rw[0]);
  store_lds(tiles[0], ra[0], rw[0]);
  load_global(BK, ra[0], rw[0]);
  __syncthreads();
  // tile t is in LDS buffer t % 2; while it is worked on, tile t + 1 waits in one register set and tile t + 2 is on its
  // way into the other; a buffer is written again only after the barrier behind its last reader
  // (an odd number of tiles is worked on as the next even one: loads beyond the inner size give zeros)
  for (int t = 0; t < n_tiles; t += 2) {
    load_global((t + 2) * BK, ra[1], rw[1]);
    compute(tiles[0]);
    store_lds(tiles[1], ra[0], rw[0]);
    __syncthreads();
    load_global((t + 3) * BK, ra[0], rw[0]);
    compute(tiles[1]);
    store_lds(tiles[0], ra[1], rw[1]);
    __syncthreads();
  }
  // a lane holds column lane % 32 of a block and its rows (i / 4) * 8 + (lane / 32) * 4 + i % 4
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = wr + m * 32 + (i / 4) * 8 + (lane / 32) * 4 + i % 4;
      if (srcs[row] < 0) continue;
      bf16* y = Y + (size_t)(tile * TBM + row) * ldy;
      if (GLU) {
        const float w = pair_w[row];
#pragma unroll
        for (int n = 0; n < NT / 2; ++n) {
          const int col = col0 + wc[n] + lane % 32;
          if (col < O) y[col] = (bf16)(activate(w * acc[m][n][i], act) * (w * acc[m][NT / 2 + n][i]));
        }
      } else {
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int col = col0 + wc[n] + lane % 32;
          if (col < O) y[col] = (bf16)acc[m][n][i];
        }
      }
    }
}

template <bool GLU, int BK, int BN, int NW>
int launch_tiled_as(const bf16* X, long ldx, int top, const int* sorted_pair, const int* tile_expert, int tiles, const bf16* wa, const bf16* wb,
                    long stride, bf16* Y, long ldy, int O, int I, int act, const float* in_weight, hipStream_t stream) {
  constexpr int LDS = 2 * (int)sizeof(MoeTile<BK, BN>) + 2 * TBM * (int)sizeof(int);
  static bool prepared = false;    // (one flag per instantiation)
  if (!prepared) {
    hipError_t e = hipFuncSetAttribute((const void*)moe_gemm_tiled_kernel<GLU, BK, BN, NW>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (e != hipSuccess) return gibbs_fail("moe_gemm: %s", hipGetErrorString(e));
    prepared = true;
  }
  moe_gemm_tiled_kernel<GLU, BK, BN, NW><<<dim3(ceil_div(O, GLU ? BN / 2 : BN), tiles), NW * WAVE, LDS, stream>>>(X, ldx, top, sorted_pair, tile_expert, wa, wb,
                                                                                                        stride, Y, ldy, O, I, act, in_weight);
  return 0;
}
// Many pairs and whole tiles of k (an inner size that is a multiple of 64, two tiles or more): the same product with loads that go
// from memory to LDS without passing through registers (buffer_to_lds), three tiles deep.  An item is 128 places
// x 256 rows of W, a wave of the 8 takes 64 x 64 of it; a compute unit has one workgroup, which goes on from item to item and has
// the next one's first tiles under way while it finishes this one.  A tile in LDS is [row][64] with the 16-byte chunk c of row r at
// position c ^ ((r >> 1) & 7), so that the operand reads (32 rows x one chunk an instruction) are free of bank conflicts; the lane
// that fills a position asks memory for the chunk that belongs there.  The product is computed transposed (features x places): a
// lane's results are 4 neighbouring features of one place.
// A tile of k takes 1.0 us; alone its loads take 0.79, its matrix instructions 0.58 and its LDS reads 0.41 (128 bytes a cycle; products and reads together
// 0.81), and neither the order of the items over the XCDs nor where in k an item begins changes that.  The loads are buffer loads: with global
// ones the compiler waited for the reads of the next products in front of these (8,412 pairs of 16 experts, width 2,048, 1,024 features: gated
// 104 us, down 60, now 101 and 58; 16,384 pairs, width 4,096, 2,048 features 575 and 312, now 553 and 300, 1.0 PFLOP/s; 1,400 pairs of 8 experts,
// width 2,048, 512 features 30 and 14, now 28 and 13; 2,400 pairs of 16 experts, 1,024 features, are the other way round, gated 43.6 and down 25.7, now 43.4 and 27.1).  The kernel above takes 164 and 93, 799 and 400, 70 and 23.  Slower: a workgroup an item (122 us
// where this took 114 in the first of these), tiles of 32 k with two workgroups a compute unit (133: requests of 64 bytes), and 128 rows of W (148).
constexpr int ASYNC_BK = 64, ASYNC_BN = 256, ASYNC_STAGES = 3, ASYNC_UNITS = 256;   // (units: one workgroup a compute unit)

// v <- activate(w * v): the activation is chosen once, not for each of the 16
__device__ __forceinline__ void activate_all(floatx16& v, float w, int act) {
  auto all = [&](auto f) {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = f(w * v[i]);
  };
  switch (act) {
    case ACT_GELU_TANH: return all([](float g) { return activate(g, ACT_GELU_TANH); });
    case ACT_GELU: return all([](float g) { return activate(g, ACT_GELU); });
    case ACT_RELU: return all([](float g) { return activate(g, ACT_RELU); });
    case ACT_RELU_SQUARED: return all([](float g) { return activate(g, ACT_RELU_SQUARED); });
    default: return all([](float g) { return activate(g, ACT_SILU); });
  }
}
template <bool GLU>
__global__ __launch_bounds__(512) void moe_gemm_async_kernel(const bf16* __restrict__ X, long ldx, int top, const int* __restrict__ sorted_pair,
                                                             const int* __restrict__ tile_expert, const bf16* __restrict__ Wa,
                                                             const bf16* __restrict__ Wb, long expert_stride, bf16* __restrict__ Y, long ldy,
                                                             int O, int I, int act, const float* __restrict__ in_weight, int columns, int items) {
  constexpr int THREADS = 512, WN = 4, NB = 2, BK = ASYNC_BK, BN = ASYNC_BN, STAGES = ASYNC_STAGES, COLS = GLU ? BN / 2 : BN;
  constexpr int CPR = BK / 8;                                              // chunks of a row
  constexpr int CA = TBM * CPR / THREADS, CW = BN * CPR / THREADS, LOADS = CA + CW;   // of a thread and tile of k
  constexpr int A_ELEMS = TBM * BK, STAGE_ELEMS = (TBM + BN) * BK;
  extern __shared__ __attribute__((aligned(16))) char moe_lds[];
  bf16* tiles = (bf16*)moe_lds;                                            // [STAGES][places, then rows of W][BK]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  auto swz = [](int row) { return (row >> 1) & 7; };
  // An item is a tile of places and a block of columns; tiles without an expert stand behind all others.
  auto there = [&](int item) { return item < items && tile_expert[item / columns] >= 0; };
  // What this thread brings of an item's tile of k: chunk (tid % CPR) ^ swz(r) of row r = tid / CPR + i * THREADS / CPR.  A place
  // without a pair repeats row 0 and a row of W past the last one the last: their results are not stored.
  // (Bytes from X's, the tile's or the matrix's beginning.)
  struct Source {
    const bf16* x;
    uint32_t at[LOADS];
    int expert;
  } from, from_next;
  auto rows_of = [&](int item, Source& f) {
    const int tile = item / columns, col0 = item % columns * COLS;
    f.expert = tile_expert[tile];
    f.x = top > 0 ? X : X + (size_t)tile * TBM * ldx;
#pragma unroll
    for (int i = 0; i < CA; ++i) {
      const int r = (tid + i * THREADS) / CPR, pair = sorted_pair[tile * TBM + r];
      const int src = pair < 0 ? 0 : (top > 0 ? pair / top : r);
      f.at[i] = ((uint32_t)src * (uint32_t)ldx + ((tid % CPR) ^ swz(r)) * 8) * 2;
    }
#pragma unroll
    for (int i = 0; i < CW; ++i) {
      const int r = (tid + i * THREADS) / CPR;
      const int col = min(col0 + (GLU ? r % COLS : r), O - 1);
      f.at[CA + i] = ((uint32_t)col * (uint32_t)I + ((tid % CPR) ^ swz(r)) * 8) * 2;
    }
  };
  int item = blockIdx.x;
  if (!there(item)) return;
  rows_of(item, from);
  const int n_tiles = I / BK;                                              // (at least two)
  // (W's rows follow the places in a stage, and the lanes' slots follow each other: load i fills chunks i * THREADS on)
  // (buffer loads: a scalar base and step along k and one 32-bit offset a lane, so no vector instructions for addresses; and the compiler counts LDS reads beside
  // them, where beside the global ones it waits for all of them)
  static_assert(COLS % (THREADS / CPR) == 0, "a load's rows belong to one matrix");
  auto load_one = [&](const Source& f, int k, int buf, int i) {
    const bf16* base = i < CA ? f.x : ((GLU && (i - CA) * (THREADS / CPR) >= COLS) ? Wb : Wa) + (size_t)f.expert * expert_stride;
    buffer_to_lds(base, ~0u, k * 2, f.at[i], tiles + buf * STAGE_ELEMS + (wave * WAVE + i * THREADS) * 8);
  };
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t)
#pragma unroll
    for (int i = 0; i < LOADS; ++i) load_one(from, t * BK, t, i);
  const int wr = (wave / WN) * 64, r32 = lane % 32, h = lane / 32;
  // the wave's blocks of 32 rows of W: neighbours, or the same features of gate (first half of its blocks) and up (second half)
  int wc[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n)
    wc[n] = GLU ? (n / (NB / 2)) * COLS + (wave % WN) * (COLS / WN) + (n % (NB / 2)) * 32 : (wave % WN) * (BN / WN) + n * 32;
  constexpr int STEPS = BK / 16;
  static_assert(STEPS % 2 == 0 && STAGES == 3, "the operands' two sets take turns; two tiles of k ahead");
  const bool wide = ldy % 4 == 0 && O % 4 == 0 && ((uintptr_t)Y % 8) == 0;
  int buf = 0;
  while (true) {
    const int following = item + gridDim.x;
    const bool more = there(following);
    rows_of(more ? following : item, from_next);         // (none: this item's first tiles are asked for once more)
    floatx16 acc[NB][2];
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[n][m][i] = 0.f;
    bf16x8 fa[2][2] = {}, fw[2][NB] = {};                // (zero: the first step's products stand before any operands)
    auto products = [&](const bf16x8 (&a)[2], const bf16x8 (&w)[NB]) {
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int m = 0; m < 2; ++m) acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[n], a[m], acc[n][m], 0, 0, 0);
    };
    auto tile_of_k = [&](const Source& ahead, int k_ahead) {
      // this thread's part of the tile has landed (the barrier covers the others'); the next tile's may be on their way
      barrier_behind_loads<(STAGES - 2) * LOADS>();
      const int fill = buf == 0 ? STAGES - 1 : buf - 1;  // the buffer of the tile before, which everyone has left
      const bf16* cA = tiles + buf * STAGE_ELEMS;
      const bf16* cW = cA + A_ELEMS;
      // a step's operands are asked for before the products of the step before, the first step's before the last one's of the
      // tile before: left to the compiler each step waits for its own reads
#pragma unroll
      for (int kk = 0; kk < STEPS; ++kk) {
        const int chunk = kk * 2 + h, next = kk % 2, now = 1 - next;
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const int row = wr + m * 32 + r32;
          fa[next][m] = *(const bf16x8*)(cA + row * BK + ((chunk ^ swz(row)) << 3));
        }
#pragma unroll
        for (int n = 0; n < NB; ++n) {
          const int row = wc[n] + r32;
          fw[next][n] = *(const bf16x8*)(cW + row * BK + ((chunk ^ swz(row)) << 3));
        }
        __builtin_amdgcn_sched_barrier(0);
        products(fa[now], fw[now]);
#pragma unroll
        for (int i = kk * LOADS / STEPS; i < (kk + 1) * LOADS / STEPS; ++i) load_one(ahead, k_ahead, fill, i);
        __builtin_amdgcn_sched_barrier(0);
      }
      buf = buf == STAGES - 1 ? 0 : buf + 1;
    };
    for (int t = 0; t < n_tiles - 2; ++t) tile_of_k(from, (t + 2) * BK);
    tile_of_k(from_next, 0);
    tile_of_k(from_next, BK);
    products(fa[(STEPS - 1) % 2], fw[(STEPS - 1) % 2]);
    // a lane holds place lane % 32 of a block and features (v / 4) * 8 + (lane / 32) * 4 + v % 4
    const int tile = item / columns, col0 = item % columns * COLS;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int place = tile * TBM + wr + m * 32 + r32, pair = sorted_pair[place];
      if (pair < 0) continue;
      bf16* y = Y + (size_t)place * ldy;
      if constexpr (GLU) {
        const float w = in_weight ? in_weight[pair] : 1.f;
        activate_all(acc[0][m], w, act);
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[0][m][i] *= w * acc[1][m][i];
      }
#pragma unroll
      for (int n = 0; n < (GLU ? NB / 2 : NB); ++n)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int col = col0 + wc[n] + q * 8 + h * 4;
          bf16x4 v;
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = (bf16)acc[n][m][q * 4 + i];
          if (wide && col < O) {
            *(bf16x4*)(y + col) = v;
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (col + i < O) y[col + i] = v[i];
          }
        }
    }
    if (!more) break;
    item = following;
    from = from_next;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // nothing may still be writing LDS when the workgroup ends
}

template <bool GLU>
int launch_async(const bf16* X, long ldx, int top, const int* sorted_pair, const int* tile_expert, int tiles, const bf16* wa, const bf16* wb,
                 long stride, bf16* Y, long ldy, int O, int I, int act, const float* in_weight, hipStream_t stream) {
  constexpr int LDS = ASYNC_STAGES * (TBM + ASYNC_BN) * ASYNC_BK * (int)sizeof(bf16);
  static bool prepared = false;    // (one flag per instantiation)
  if (!prepared) {
    hipError_t e = hipFuncSetAttribute((const void*)moe_gemm_async_kernel<GLU>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (e != hipSuccess) return gibbs_fail("moe_gemm: %s", hipGetErrorString(e));
    prepared = true;
  }
  const int columns = ceil_div(O, GLU ? ASYNC_BN / 2 : ASYNC_BN);
  GIBBS_REQUIRE((long)columns * tiles < (1L << 30), "moe_gemm: %d columns of %d tiles", columns, tiles);
  moe_gemm_async_kernel<GLU><<<std::min(ASYNC_UNITS, columns * tiles), 512, LDS, stream>>>(X, ldx, top, sorted_pair, tile_expert, wa, wb, stride, Y, ldy, O, I,
                                                                                    act, in_weight, columns, columns * tiles);
  return 0;
}
template <bool GLU>
int launch_tiled(const bf16* X, long ldx, int top, const int* sorted_pair, const int* tile_expert, int tiles, const bf16* wa, const bf16* wb,
                 long stride, bf16* Y, long ldy, int O, int I, int act, const float* in_weight, hipStream_t stream) {
  // Short inner sizes of one matrix stay with the kernel whose workgroups are many where the other's second or third round of items would be
  // the last and leave three eighths of the units idle or more (8,320 pairs of 16 experts, us, here and there: 1,024 features, inner size 128
  // 14.5 and 17.1, 256 19.3 and 21.5, 512 28.2 and 27.1; 2,048 features, 128 23.6 and 26.3).
  const long items = (long)ceil_div(O, GLU ? ASYNC_BN / 2 : ASYNC_BN) * tiles, last = items % ASYNC_UNITS;
  const bool idle = !GLU && I < 512 && items > ASYNC_UNITS && items <= 3 * ASYNC_UNITS && last > 0 && last <= ASYNC_UNITS * 5 / 8;
  // (its loads have 32-bit offsets within X, the rows of a step, and within a matrix)
  const bool near = (top > 0 ? (long)tiles * TBM / top + 1 : TBM) * ldx < (1L << 31) && (long)O * I < (1L << 31);
  if (I % ASYNC_BK == 0 && I >= 2 * ASYNC_BK && !idle && near)
    return launch_async<GLU>(X, ldx, top, sorted_pair, tile_expert, tiles, wa, wb, stride, Y, ldy, O, I, act, in_weight, stream);
  // what is left: wide results with a long inner size 256 rows of W a workgroup and 8 waves (the tile of X is read by half as many
  // workgroups: 8,320 pairs, 2,048 features, inner size 2,056 gated 264 us, with 128 rows 306); otherwise 128 rows and 4 waves, which leaves
  // more workgroups to spread
  if (I > 1024 && O >= 512)
    return launch_tiled_as<GLU, 32, 256, 8>(X, ldx, top, sorted_pair, tile_expert, tiles, wa, wb, stride, Y, ldy, O, I, act, in_weight, stream);
  return launch_tiled_as<GLU, 32, 128, 4>(X, ldx, top, sorted_pair, tile_expert, tiles, wa, wb, stride, Y, ldy, O, I, act, in_weight, stream);
}

// ------------------------------------------------------------------------------------------------- combine
// (`self` [n, W], not null: a choice whose place is -1 is an identity expert, its result the row of `self`)
template <typename T, bool VEC>
__global__ void moe_combine_kernel(const T* __restrict__ y, const int* __restrict__ pair_pos, const float* __restrict__ weight,
                                   const T* __restrict__ shared, const float* __restrict__ sgate, const T* __restrict__ self,
                                   T* __restrict__ out, int top, int W) {
  constexpr int MOST = 8;      // choices whose places and weights a thread keeps in registers
  const int n = blockIdx.x;
  const float g = shared ? (sgate ? sgate[n] : 1.0f) : 0.f;
  const T* at[MOST];
  float w[MOST];
  auto row_of = [&](int s) -> const T* {
    const int place = pair_pos[(size_t)n * top + s];
    return (self && place < 0) ? self + (size_t)n * W : y + (size_t)place * W;
  };
#pragma unroll
  for (int s = 0; s < MOST; ++s) {
    at[s] = s < top ? row_of(s) : y;
    w[s] = s < top ? (weight ? weight[(size_t)n * top + s] : 1.f) : 0.f;
  }
  if (VEC) {
    for (int c = threadIdx.x * 4; c < W; c += blockDim.x * 4) {
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int s = 0; s < MOST; ++s)
        if (s < top) {
          const float4 r = load4f(at[s] + c);
          v.x = fmaf(w[s], r.x, v.x); v.y = fmaf(w[s], r.y, v.y); v.z = fmaf(w[s], r.z, v.z); v.w = fmaf(w[s], r.w, v.w);
        }
      for (int s = MOST; s < top; ++s) {
        const float ws = weight ? weight[(size_t)n * top + s] : 1.f;
        const float4 r = load4f(row_of(s) + c);
        v.x = fmaf(ws, r.x, v.x); v.y = fmaf(ws, r.y, v.y); v.z = fmaf(ws, r.z, v.z); v.w = fmaf(ws, r.w, v.w);
      }
      if (shared) {
        const float4 r = load4f(shared + (size_t)n * W + c);
        v.x = fmaf(g, r.x, v.x); v.y = fmaf(g, r.y, v.y); v.z = fmaf(g, r.z, v.z); v.w = fmaf(g, r.w, v.w);
      }
      store4f(out + (size_t)n * W + c, v);
    }
    return;
  }
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    float v = 0.f;
    for (int s = 0; s < top; ++s) v = fmaf(weight ? weight[(size_t)n * top + s] : 1.f, to_float(row_of(s)[c]), v);
    if (shared) v = fmaf(g, to_float(shared[(size_t)n * W + c]), v);
    out[(size_t)n * W + c] = from_float<T>(v);
  }
}
}  // namespace

// Places that the sorted pairs of a step can take at most: every expert's stretch rounded up to whole tiles.
GIBBS_EXPORT long gibbs_moe_capacity(int n_pairs, int E, int bm) {
  return ((long)n_pairs + (long)E * (bm - 1) + bm - 1) / bm * bm;
}
// Tiles of pairs: 16 while the matrices are streamed for few pairs each (at most 64 an expert on average), 128 beyond.
GIBBS_EXPORT int gibbs_moe_tile(int n_pairs, int E) { return (long)n_pairs <= 64L * E ? 16 : 128; }

// Features of a workgroup of the gated product of few pairs, in `tiles` tiles at most (those that no expert takes among them): 16 while they give the chip no more than
// ten workgroups a compute unit, 32 beyond, where the rows of X and the features that several tiles share come from the L2s and are read less often so.
// 32 / 16, us: 16 experts of 1,024 at width 2,048, 4 chosen, 32 rows (1,472 workgroups of 16) 30.6 / 28.7, 96 (2,496) 44.5 / 45.1, 128 (3,008) 50.3 / 55.2, 256 90.2 / 98.9;
// of 512 at 1,024 192 rows (2,016) 24.1 / 22.9, 256 (2,528) 28.5 / 29.1; 8 of 1,024 at 1,024, 2 chosen, 256 rows (2,528) 28.3 / 27.8; 64 of 512 at 2,048, 8 chosen, 96 rows
// (3,456) 59.9 / 54.5, 128 65.4 / 66.6, 235 (5,664) 88 / 98, 512 167 / 191.
GIBBS_EXPORT int gibbs_moe_gated_features(int tiles, int F) { return (long)tiles * ceil_div(F, 16) <= 2560 ? 16 : 32; }

// Few rows, whose products need no grouping (gibbs_moe_gemm_direct): at most 16, so that an expert has at most one of each row's pairs, a tile, and
// 64 pairs, one for each lane of a wave.  Any number of experts: a grid of grouped products has a workgroup for the tile that each may begin, as this one has for each.
// Route, group and products grouped / without grouping, us, width 2,048, F 1,024, 4 chosen, 8 rows: 16 experts 48 / 50, 64 87 / 86, 256 133 / 135, 512 177 / 165, 1,024
// 304 / 272; 1 row: 64 31 / 32, 256 66 / 59, 1,024 215 / 169; width 1,024, F 512, 8 rows: 16 22 / 19, 256 58 / 51, 1,024 153 / 110.
GIBBS_EXPORT int gibbs_moe_direct_takes(int n, int top, int E, int W, int F) {
  return n > 0 && n <= 16 && n * top <= WAVE && E <= 65535 && W % 8 == 0 && F % 8 == 0;
}

// mode 0: the largest logits (+ bias), weights by the softmax over the chosen; mode 1: scores by the softmax over all E
// outputs, the largest of score + router_bias (a correction that only the choice sees), weights the chosen scores over their sum;
// mode 2: scores by the sigmoid of every output alone, the largest of score + router_bias, weights the chosen scores.
// weight_scale: mode 1's weights times a constant.
GIBBS_EXPORT int gibbs_moe_route_scaled(const void* h, long ldh, int dtype, const float* router, const float* router_bias,
                                        const float* shared_gate, int* chosen, float* weight, float* sgate, int n, int W, int E, int top,
                                        int mode, float weight_scale, hipStream_t stream) {
  return gibbs_moe_route_placed(h, ldh, dtype, router, router_bias, shared_gate, chosen, weight, sgate, nullptr, 0, n, W, E, top, mode, weight_scale, stream);
}
// The same, and for products without grouping place [n, top] (null: none): the pair's own number, or -1 where its choice is none of the
// first `matrices` (an identity expert).  At most 1,023 rows and 64 choices.
GIBBS_EXPORT int gibbs_moe_route_placed(const void* h, long ldh, int dtype, const float* router, const float* router_bias,
                                        const float* shared_gate, int* chosen, float* weight, float* sgate, int* place, int matrices, int n, int W, int E, int top,
                                        int mode, float weight_scale, hipStream_t stream) {
  GIBBS_REQUIRE(!place || (n < 1024 && top <= WAVE), "moe_route: places for %d rows of %d choices", n, top);
  GIBBS_REQUIRE(weight_scale == 1.0f || mode == 1, "moe_route: weights times %g go with the scores' softmax over all outputs", weight_scale);
  GIBBS_REQUIRE(mode >= 0 && mode <= 2, "moe_route: mode %d", mode);
  GIBBS_REQUIRE(h && router && chosen && weight && n > 0 && W > 0 && ldh >= W, "moe_route: bad operands n=%d width=%d", n, W);
  GIBBS_REQUIRE(E > 0 && E <= MOE_MAX_EXPERTS && top > 0 && top <= E, "moe_route: %d of %d experts (at most %d)", top, E, MOE_MAX_EXPERTS);
  GIBBS_REQUIRE(!shared_gate || sgate, "moe_route: a shared expert's gate needs its output");
  const size_t lds = (size_t)E * sizeof(float) * (mode != 0 ? 2 : 1);
  // few rows: a wave per expert (and one for the shared expert's gate) up to 16 waves; many rows fill the chip with 4; more share the router.
  // A row / four rows a workgroup, us, where the line lies: 8 experts 1,280 rows of 1,024 13.0 / 13.6, 1,536 13.8 / 13.7, of 256 12.7 / 12.5, of 2,048 768
  // 13.0 / 13.0, 1,024 13.6 / 12.9; 32 experts 1,024 rows of 1,024 18.2 / 20.4, 1,536 24.5 / 22.5, of 512 21.8 / 20.1, of 2,048 768 22.6 / 23.0, 1,024 26.0 /
  // 23.1; 64 experts 1,536 rows of 1,024 38.3 / 33.4, 1,024 of 2,048 41.6 / 36.3, 4,096 127 / 62; 256 experts 1,024 rows of 2,048 138 / 120, 4,096 484 / 206,
  // 512 experts 1,024 rows 264 / 272
  const bool share = (n >= 1536 || (n >= 1024 && W >= 2048)) && E <= 256 && W % 4 == 0 && ldh % 4 == 0 && ((uintptr_t)h % 16) == 0 && ((uintptr_t)router % 16) == 0 && ((uintptr_t)shared_gate % 16) == 0;
  if (share && (dtype == GIBBS_F32 || dtype == GIBBS_BF16)) {
    const int blocks = ceil_div(n, ROUTE_ROWS);
    const size_t all = 2 * ROUTE_ROWS * (size_t)E * sizeof(float);
    if (dtype == GIBBS_F32)
      moe_route_rows_kernel<float><<<blocks, ROUTE_ROWS * WAVE, all, stream>>>((const float*)h, ldh, router, router_bias, shared_gate, chosen, weight, sgate, n, W, E, top, mode, weight_scale);
    else
      moe_route_rows_kernel<bf16><<<blocks, ROUTE_ROWS * WAVE, all, stream>>>((const bf16*)h, ldh, router, router_bias, shared_gate, chosen, weight, sgate, n, W, E, top, mode, weight_scale);
    GIBBS_LAUNCH_STATUS("moe_route");
  }
  const int threads = n >= 512 ? 256 : WAVE * std::min(16, std::max(4, E + 1));
  if (dtype == GIBBS_F32)
    moe_route_kernel<float><<<n, threads, lds, stream>>>((const float*)h, ldh, router, router_bias, shared_gate, chosen, weight, sgate, W, E, top, mode, weight_scale, place, matrices);
  else if (dtype == GIBBS_BF16)
    moe_route_kernel<bf16><<<n, threads, lds, stream>>>((const bf16*)h, ldh, router, router_bias, shared_gate, chosen, weight, sgate, W, E, top, mode, weight_scale, place, matrices);
  else
    return gibbs_fail("moe_route: unknown dtype %d", dtype);
  GIBBS_LAUNCH_STATUS("moe_route");
}
GIBBS_EXPORT int gibbs_moe_route_mode(const void* h, long ldh, int dtype, const float* router, const float* router_bias,
                                      const float* shared_gate, int* chosen, float* weight, float* sgate, int n, int W, int E, int top,
                                      int mode, hipStream_t stream) {
  return gibbs_moe_route_scaled(h, ldh, dtype, router, router_bias, shared_gate, chosen, weight, sgate, n, W, E, top, mode, 1.0f, stream);
}
GIBBS_EXPORT int gibbs_moe_route(const void* h, long ldh, int dtype, const float* router, const float* router_bias,
                                 const float* shared_gate, int* chosen, float* weight, float* sgate, int n, int W, int E, int top,
                                 hipStream_t stream) {
  return gibbs_moe_route_mode(h, ldh, dtype, router, router_bias, shared_gate, chosen, weight, sgate, n, W, E, top, 0, stream);
}

GIBBS_EXPORT int gibbs_moe_group(const int* chosen, int n_pairs, int E, int bm, int* sorted_pair, int* pair_pos, int* tile_expert,
                                 long cap, hipStream_t stream) {
  GIBBS_REQUIRE(chosen && sorted_pair && pair_pos && tile_expert && n_pairs > 0, "moe_group: bad operands pairs=%d", n_pairs);
  GIBBS_REQUIRE(E > 0 && E <= MOE_MAX_EXPERTS && (bm == 16 || bm == 128), "moe_group: %d experts (at most %d) in tiles of %d (16 or 128)", E, MOE_MAX_EXPERTS, bm);
  GIBBS_REQUIRE(cap >= gibbs_moe_capacity(n_pairs, E, bm) && cap % bm == 0 && cap < (1L << 31), "moe_group: %ld places for %d pairs of %d experts", cap, n_pairs, E);
  moe_group_kernel<<<1, 1024, 0, stream>>>(chosen, n_pairs, E, bm, sorted_pair, pair_pos, tile_expert, (int)cap);
  GIBBS_LAUNCH_STATUS("moe_group");
}

// Rows of 4 KB and more are read from a k of the features' own on; a loop that can turn costs shorter ones more than it gives (8 rows of 16 experts of 512 at width
// 1,024, gated, us: 8.74, 9.12 with a turn of none).
static bool few_turns(int I) { return I >= 2048; }

// Y[m] = W_a,e X[src(m)] (w_b null), or act(W_a,e X[src(m)]) * (W_b,e X[src(m)]), for every place m of the sorted pairs; e the
// expert of m's tile; src(m) = pair / top (top > 0: rows of the step, gathered) or m itself (top 0: X is in sorted order).
// W_a, W_b: [experts, O, I].
// in_weight [pairs] (null: 1; with w_b only): both products of a place are multiplied by its pair's weight before the activation.
GIBBS_EXPORT int gibbs_moe_gemm(const void* X, long ldx, int top, const int* sorted_pair, const int* tile_expert, long cap, int bm,
                                const void* w_a, const void* w_b, void* Y, long ldy, int dtype, int O, int I, int act,
                                hipStream_t stream) {
  return gibbs_moe_gemm_weighted(X, ldx, top, sorted_pair, tile_expert, cap, bm, w_a, w_b, nullptr, Y, ldy, dtype, O, I, act, stream);
}
GIBBS_EXPORT int gibbs_moe_gemm_weighted(const void* X, long ldx, int top, const int* sorted_pair, const int* tile_expert, long cap, int bm,
                                         const void* w_a, const void* w_b, const float* in_weight, void* Y, long ldy, int dtype, int O, int I,
                                         int act, hipStream_t stream) {
  GIBBS_REQUIRE(!in_weight || w_b, "moe_gemm: weights on the inputs go with the gated products");
  GIBBS_REQUIRE(X && sorted_pair && tile_expert && w_a && Y && O > 0 && I > 0 && ldx >= I && ldy >= O, "moe_gemm: bad operands O=%d I=%d", O, I);
  GIBBS_REQUIRE((bm == 16 || bm == 128) && cap > 0 && cap % bm == 0 && cap / bm <= 65535, "moe_gemm: %ld places in tiles of %d", cap, bm);
  GIBBS_REQUIRE(top >= 0 && act >= 0 && act < ACT_COUNT, "moe_gemm: bad choice count or activation");
  const long stride = (long)O * I;
  const int tiles = (int)(cap / bm);
#define MOE_PLAIN(T, BM, GLU)                                                                                                     \
  moe_gemm_plain_kernel<T, BM, GLU><<<dim3(ceil_div(O, 64), tiles), 256, 0, stream>>>((const T*)X, ldx, top, sorted_pair, tile_expert, \
                                                                                     (const T*)w_a, (const T*)w_b, stride, (T*)Y, ldy, O, I, act, in_weight)
#define MOE_PLAIN_ANY(T)                                                                  \
  do {                                                                                    \
    if (bm == 128) { if (w_b) MOE_PLAIN(T, 128, true); else MOE_PLAIN(T, 128, false); }    \
    else { if (w_b) MOE_PLAIN(T, 16, true); else MOE_PLAIN(T, 16, false); }                \
  } while (0)
  if (dtype == GIBBS_F32) {
    if (!moe_gemm_f32((const float*)X, ldx, top, sorted_pair, tile_expert, cap, bm, (const float*)w_a, (const float*)w_b, in_weight, (float*)Y, ldy, O, I, act, stream))
      MOE_PLAIN_ANY(float);
  } else if (dtype == GIBBS_BF16) {
    const bool aligned = I % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)X % 16) == 0 && ((uintptr_t)w_a % 16) == 0 && ((uintptr_t)w_b % 16) == 0;
    if (!aligned) {
      MOE_PLAIN_ANY(bf16);
    } else if (bm == 128) {
      if (w_b ? launch_tiled<true>((const bf16*)X, ldx, top, sorted_pair, tile_expert, tiles, (const bf16*)w_a, (const bf16*)w_b, stride, (bf16*)Y, ldy, O, I, act, in_weight, stream)
              : launch_tiled<false>((const bf16*)X, ldx, top, sorted_pair, tile_expert, tiles, (const bf16*)w_a, nullptr, stride, (bf16*)Y, ldy, O, I, act, nullptr, stream))
        return 1;
    } else if (w_b) {
      const auto queue = [&](auto kernel, int features) {
        kernel<<<dim3(ceil_div(O, features), tiles), 256, 0, stream>>>((const bf16*)X, sorted_pair, tile_expert, (const bf16*)w_a, (const bf16*)w_b, top, I, ldx, stride, (bf16*)Y,
                                                                       ldy, O, act, in_weight, 0, 0);
      };
      const bool narrow = gibbs_moe_gated_features(tiles, O) == 16;
      if (few_turns(I)) narrow ? queue(moe_gemm_few_kernel<true, false, 1, true>, 16) : queue(moe_gemm_few_kernel<true, false, 2, true>, 32);
      else narrow ? queue(moe_gemm_few_kernel<true, false, 1, false>, 16) : queue(moe_gemm_few_kernel<true, false, 2, false>, 32);
    } else {
      const auto kernel = few_turns(I) ? moe_gemm_few_kernel<false, false, 2, true> : moe_gemm_few_kernel<false, false, 2, false>;
      kernel<<<dim3(ceil_div(O, 32), tiles), 256, 0, stream>>>((const bf16*)X, sorted_pair, tile_expert, (const bf16*)w_a, nullptr, top, I, ldx, stride, (bf16*)Y, ldy, O, act,
                                                               nullptr, 0, 0);
    }
  } else {
    return gibbs_fail("moe_gemm: unknown dtype %d", dtype);
  }
#undef MOE_PLAIN_ANY
#undef MOE_PLAIN
  GIBBS_LAUNCH_STATUS("moe_gemm");
}

// The products of few rows (gibbs_moe_direct_takes) straight from their choices `chosen` [pairs], bfloat16: row i of Y is pair i's result; X's rows are the step's
// (gated: w_b given, row pair / top) or the pairs' own (w_b null).  Choices of E and beyond have no result.
GIBBS_EXPORT int gibbs_moe_gemm_direct(const void* X, long ldx, int top, const int* chosen, int pairs, int E, const void* w_a, const void* w_b,
                                       const float* in_weight, void* Y, long ldy, int O, int I, int act, hipStream_t stream) {
  GIBBS_REQUIRE(X && chosen && w_a && Y && O > 0 && I > 0 && ldx >= I && ldy >= O && top > 0, "moe_gemm: bad operands O=%d I=%d", O, I);
  GIBBS_REQUIRE(pairs > 0 && pairs <= WAVE && pairs % top == 0 && pairs / top <= 16 && E > 0 && E <= 65535, "moe_gemm: %d pairs of %d a row without grouping", pairs, top);
  GIBBS_REQUIRE(act >= 0 && act < ACT_COUNT && (!in_weight || w_b), "moe_gemm: bad activation, or weights on the inputs of an ungated product");
  GIBBS_REQUIRE(I % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)X % 16) == 0 && ((uintptr_t)w_a % 16) == 0 && ((uintptr_t)w_b % 16) == 0, "moe_gemm: rows of whole 16 bytes");
  const long stride = (long)O * I;
  const int chosen_experts = std::min(E, pairs);      // (at most)
  if (w_b) {
    const auto kernel = few_turns(I) ? moe_gemm_few_kernel<true, true, 1, true> : moe_gemm_few_kernel<true, true, 1, false>;
    kernel<<<dim3(ceil_div(O, 16), chosen_experts), 256, 0, stream>>>((const bf16*)X, chosen, nullptr, (const bf16*)w_a, (const bf16*)w_b, top, I, ldx, stride, (bf16*)Y, ldy, O, act,
                                                                      in_weight, pairs, E);
  } else {
    const auto kernel = few_turns(I) ? moe_gemm_few_kernel<false, true, 2, true> : moe_gemm_few_kernel<false, true, 2, false>;
    kernel<<<dim3(ceil_div(O, 32), chosen_experts), 256, 0, stream>>>((const bf16*)X, chosen, nullptr, (const bf16*)w_a, nullptr, 0, I, ldx, stride, (bf16*)Y, ldy, O, act, nullptr,
                                                                      pairs, E);
  }
  GIBBS_LAUNCH_STATUS("moe_gemm");
}

// out[n] = sum_c weight[n][c] y[pair_pos[n * top + c]] + sgate[n] shared[n]  (shared null: no shared expert; sgate or weight null: 1).
GIBBS_EXPORT int gibbs_moe_combine(const void* y, const int* pair_pos, const float* weight, const void* shared, const float* sgate,
                                   void* out, int dtype, int n, int top, int W, hipStream_t stream) {
  return gibbs_moe_combine_self(y, pair_pos, weight, shared, sgate, nullptr, out, dtype, n, top, W, stream);
}
// self [n, W] (null: none): the rows themselves, which a choice without a place (-1: an identity expert) stands for.
GIBBS_EXPORT int gibbs_moe_combine_self(const void* y, const int* pair_pos, const float* weight, const void* shared, const float* sgate,
                                        const void* self, void* out, int dtype, int n, int top, int W, hipStream_t stream) {
  GIBBS_REQUIRE(y && pair_pos && out && n > 0 && top > 0 && W > 0, "moe_combine: bad operands n=%d top=%d width=%d", n, top, W);
  const size_t bytes = dtype == GIBBS_F32 ? 16 : 8;
  const bool vec = W % 4 == 0 && ((uintptr_t)y % bytes) == 0 && ((uintptr_t)shared % bytes) == 0 && ((uintptr_t)out % bytes) == 0 && ((uintptr_t)self % bytes) == 0;
  const int threads = vec ? (W >= 4096 ? 1024 : (W >= 1024 ? 256 : 64)) : (W >= 1024 ? 256 : 64);
#define MOE_COMBINE(T, V) moe_combine_kernel<T, V><<<n, threads, 0, stream>>>((const T*)y, pair_pos, weight, (const T*)shared, sgate, (const T*)self, (T*)out, top, W)
  if (dtype == GIBBS_F32) {
    if (vec) MOE_COMBINE(float, true); else MOE_COMBINE(float, false);
  } else if (dtype == GIBBS_BF16) {
    if (vec) MOE_COMBINE(bf16, true); else MOE_COMBINE(bf16, false);
  } else
    return gibbs_fail("moe_combine: unknown dtype %d", dtype);
  GIBBS_LAUNCH_STATUS("moe_combine");
}
