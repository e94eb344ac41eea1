// Paged causal attention for prompt portions, head sizes 64 and 128: matrix instructions of 32 x 32, scores, weights and values side by side.
//
// A workgroup of 4 waves takes 32 RW consecutive query rows of one request and HW query heads that share a kv head (as many of the group's as
// divide 4); a wave owns 32 rows of one head.  Keys are walked in tiles of 64 aligned to absolute key index, so that in a call of one slice a row's
// sequence of operations depends neither on how the prompt was cut nor on HW (slices begin and end by the workgroup's rows).  As in attention_prefill.hip the scores are made transposed, S^T = K Q^T, and
// exp(S - m) is, as it lies in the registers, the B operand of O^T += V^T P^T, V^T by the transposing LDS read.
//
// What bounds it: the vector instructions of the softmax (per 64 keys and 32 rows some 135, 33 of them exponentials of 8 cycles: 800 cycles),
// beside 512 cycles of the matrix cores, which run at the same time only if a wave issues them in turn.  So a step works on three tiles at once:
// the weights of tile t, the scores of tile t + 1 and the values of tile t - 1, sixteen slices (head size 64) of one matrix instruction
// with the vector instructions that fit its 32 cycles, the order pinned.  Left to the compiler each kind came in a block of its own, and three
// waves a SIMD side by side did no better (16,384 rows of 32 heads: 1,373 us against 1,277).  Against 16 rows a wave, twice the products
// per byte read from LDS; K and V go from memory to LDS without registers (buffer_to_lds), 16-byte chunks of a row swapped by its number so that
// no read has a bank conflict.  The longest workgroup's chain of tiles bounds short prompts, so workgroups are 32 rows rather than 64.
// Measured, us a call, 32 heads of 64 in groups of 4, the kernel of 16 rows a wave and this one: 1,024 rows 30 and 19; 2,048 58 and 38; 4,096
// 193 and 104; 16,384 1,764 and 1,280 (860 TFLOP/s); 3 x 700 rows 28 and 19, and 16 heads of 128 31 and 24.  With the loads to LDS as buffer loads,
// beside which the compiler waits for the reads of LDS that a product needs and not for those of the next three: 2,048 rows 38.1 -> 36.7, 4,096
// 107 -> 103, 16,384 1,253 -> 1,230.
// Tiles in flight for longer (four of each in LDS): the same.
#include "attention_prompt.h"

namespace {
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;
typedef short short4v __attribute__((ext_vector_type(4)));
typedef short short8v __attribute__((ext_vector_type(8)));

constexpr int BN = 64;   // keys per tile
// (a value is made where this stands, not moved to where it is used)
#define HOLD(v) asm volatile("" : "+v"(v))

// What the other half of the wave holds of the same row, folded in: both halves get the result.
__device__ __forceinline__ float halves_max(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ float halves_sum(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}
__device__ __forceinline__ short4v lds_read_transposed(const bf16* p, int bytes) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)(const bf16*)((const char*)p + bytes));
}

// Where the 16-byte chunk c of a row (of 8 or 16) lies in LDS: at c ^ swizzle(row).
template <int HD>
__device__ __forceinline__ int key_swizzle(int row) { return HD == 64 ? (row >> 1) & 7 : row & 15; }
template <int HD>
__device__ __forceinline__ int value_swizzle(int row) { return (row & 3) << (HD == 64 ? 1 : 2); }

template <int HD, int HW, int RW, int SCORES>
__global__ __launch_bounds__(64 * HW * RW) __attribute__((amdgpu_waves_per_eu(2))) void attention_prompt_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ kpages, const bf16* __restrict__ vpages, bf16* __restrict__ out,
    float* __restrict__ partial, PrefillArgs a) {
  constexpr bool BIAS = SCORES != SCORES_PLAIN, CAP = SCORES == SCORES_CAPPED;
  constexpr int NW = HW * RW, NT = 64 * NW;
  constexpr int BM = 32 * RW;          // query rows of the workgroup
  constexpr int ND = HD / 32;          // blocks of 32 over d (the values' product)
  constexpr int DS = HD / 16;          // steps of 16 over d (the scores' product)
  constexpr int CPR = HD / 8;          // 16-byte chunks of a key
  constexpr int RPL = 64 / CPR;        // keys that one load of a wave covers
  constexpr int NI = BN / RPL / NW;    // loads of K (and of V) per wave and tile
  static_assert(NI >= 1 && NI * NW * RPL == BN, "whole loads");
  // Tiles in LDS that take turns, each an array of its own: reading one does not make the compiler wait for the loads into the others.
  __shared__ __attribute__((aligned(16))) bf16 sK0[BN * HD], sK1[BN * HD], sV0[BN * HD], sV1[BN * HD];
  constexpr int NB = BN + BM;          // (entry BM - 1 + key - row of the tile)
  __shared__ float sB[BIAS ? 2 : 1][BIAS ? HW : 1][BIAS ? NB : 1];

  const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int groups = a.nh / HW;
  // which request and which of its tiles of rows: 64 requests at a time, a lane each
  int tile = blockIdx.x / groups, r = -1, qlen = 0;
  const int head_group = blockIdx.x % groups;
  if (a.n_req == 1) {
    qlen = a.cu[1] - a.cu[0];
    const int tiles = (qlen + BM - 1) / BM;
    if (tile >= tiles) return;
    r = 0;
    tile = tiles - 1 - tile;      // a request's last rows see the most keys: those workgroups start first
  }
  for (int base = 0; r < 0 && base < a.n_req; base += WAVE) {
    const int i = min(base + lane, a.n_req - 1);
    const int len = base + lane < a.n_req ? a.cu[i + 1] - a.cu[i] : 0;
    int upto = (len + BM - 1) / BM;      // tiles of these requests up to this one
#pragma unroll
    for (int d = 1; d < WAVE; d *= 2) {
      const int before = __shfl_up(upto, d, WAVE);
      if (lane >= d) upto += before;
    }
    const unsigned long long behind = __builtin_amdgcn_ballot_w64(tile < upto);
    if (behind) {
      const int l = __builtin_ctzll(behind);
      r = base + l;
      qlen = __builtin_amdgcn_readlane(len, l);
      tile = __builtin_amdgcn_readlane(upto, l) - 1 - tile;
      break;
    }
    tile -= __builtin_amdgcn_readlane(upto, WAVE - 1);
  }
  if (r < 0) return;
  const int head = head_group * HW + wave / RW;
  const int kvh = head_group * HW / (a.nh / a.nkv);
  const int lr = lane % 32, h = lane / 32;
  const int row0 = (wave % RW) * 32;                 // the wave's first row inside the tile
  const int n0 = a.cu[r] + tile * BM;                // the tile's first row among the step's rows
  const int p0 = a.ctx[r] + tile * BM;               // its absolute position
  const int rows_here = min(BM, qlen - tile * BM);
  const int* table = a.table + (size_t)r * a.max_pages;

  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8 qf[DS];
#pragma unroll
  for (int s = 0; s < DS; ++s)
    qf[s] = row0 + lr < rows_here ? *(const bf16x8*)(q + (size_t)(n0 + row0 + lr) * a.ldq + (size_t)head * HD + s * 16 + h * 8) : zero8;
  const int my_row = min(row0 + lr, rows_here - 1);
  const int pos_row = p0 + my_row;
  const int lo_row = a.chunk > 0 ? pos_row - pos_row % a.chunk - 1 : (a.window > 0 ? pos_row - a.window : -1);

  float m = -1e30f, l = 0.f;   // maximum of the raw scores (finite while no key is seen); this lane's share of the sum
  floatx16 o[ND];
#pragma unroll
  for (int t = 0; t < ND; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[t][i] = 0.f;

  const float scale2 = a.scale * 1.44269504088896340736f;
  const int last_pos = p0 + rows_here - 1;
  auto first_of = [&](int p) { return a.chunk > 0 ? p - p % a.chunk : (a.window > 0 ? max(0, p - a.window + 1) : 0); };
  const float cap_raw = CAP ? a.softcap / a.scale : 0.f, cap_inv = CAP ? a.scale / a.softcap : 0.f;

  int kt_first = first_of(p0) / BN, kt_stop = last_pos / BN + 1;
  if (a.n_splits > 1) {
    const int per = (kt_stop - kt_first + a.n_splits - 1) / a.n_splits;
    kt_first += blockIdx.z * per;
    kt_stop = min(kt_stop, kt_first + per);
  }

  // ---- keys and values: memory -> LDS
  const size_t page_stride = (size_t)a.nkv * a.page_size * HD;
  const size_t head_off = (size_t)kvh * a.page_size * HD;
  const int lrow = lane / CPR, lslot = lane % CPR;
  int ids[NI], ids_from = kt_first;     // page ids of the wave's keys in 64 tiles, a tile a lane
  auto load_ids = [&](int kt) {
    ids_from = kt;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int key = min((kt + lane) * BN + (wave * NI + i) * RPL, last_pos);
      const int page = table[key >> a.page_shift];
      ids[i] = page < 0 ? 0 : (page >= a.num_pages ? a.num_pages - 1 : page);   // never read outside the pool
    }
  };
  auto bring = [&](const bf16* __restrict__ pages, bool values, bf16* dst, int kt) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int row = (wave * NI + i) * RPL;        // (of the tile)
      const int page = __builtin_amdgcn_readlane(ids[i], kt - ids_from);
      const int key = min(kt * BN + row, last_pos);
      const bf16* at = pages + (size_t)page * page_stride + head_off + (size_t)((unsigned)(key & (a.page_size - 1)) / RPL * RPL * HD);
      const int chunk = lslot ^ (values ? value_swizzle<HD>(row + lrow) : key_swizzle<HD>(row + lrow));
      const unsigned lane_at = (unsigned)(lrow * HD + chunk * 8) * 2;
      buffer_to_lds(at, RPL * HD * 2, 0, lane_at, dst + row * HD);
    }
  };
  // values beyond the last key: whatever the page held there, a weight of zero must not meet a NaN
  auto clear_tail = [&](bf16* dst, int kt) {
    if (kt * BN + BN - 1 <= last_pos) return;
    for (int c = tid; c < BN * CPR; c += NT)
      if (kt * BN + c / CPR > last_pos) *(uint4*)&dst[c * 8] = make_uint4(0, 0, 0, 0);
    __syncthreads();
  };
  const bool biased = BIAS && (!CAP || a.bias);
  // a bias's values go through registers, asked for a tile earlier
  constexpr int NBI = (NB * HW + NT - 1) / NT;
  float breg[NBI];
  auto ask_bias = [&](int kt) {
#pragma unroll
    for (int i = 0; i < NBI; ++i) {
      const int c = min(tid + i * NT, NB * HW - 1);
      const int back = p0 + BM - 1 - kt * BN - c % NB;
      breg[i] = a.bias[(size_t)(head_group * HW + c / NB) * a.bias_len + min(max(back, 0), a.bias_len - 1)];
    }
  };
  auto put_bias = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NBI; ++i) {
      const int c = tid + i * NT;
      if (c < NB * HW) sB[buf][c / NB][c % NB] = breg[i];
    }
  };

  // ---- S^T = K Q^T: two blocks of 32 keys; this lane gets S[row lr][key c*32 + (i/4)*8 + h*4 + i%4]
  constexpr int KA = HD == 64 ? 4 : 8;
  int k_at[KA];
#pragma unroll
  for (int s = 0; s < KA; ++s) k_at[s] = lr * HD * 2 + (((s * 2 + h) ^ key_swizzle<HD>(lr)) << 4);   // (bytes)
  auto scores = [&](const bf16* sK, floatx16 (&s2)[2]) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s2[c][i] = 0.f;
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        const bf16x8 kf = *(const bf16x8*)((const char*)sK + k_at[s] + c * 64 * HD);
        s2[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[s], s2[c], 0, 0, 0);
      }
    }
  };
  auto largest = [&](const floatx16 (&s2)[2]) {
    float mx = fmaxf(s2[0][0], s2[1][15]);
#pragma unroll
    for (int i = 1; i < 31; i += 2) mx = fmaxf(fmaxf(mx, s2[i / 16][i % 16]), s2[(i + 1) / 16][(i + 1) % 16]);
    return mx;
  };
  // what is done to raw scores before the softmax; mx, their largest, is taken again where they change
  auto shape = [&](int buf, floatx16 (&s2)[2], int key0, float& mx) {
    if constexpr (CAP) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < 16; ++i) s2[c][i] = cap_raw * tanhf(s2[c][i] * cap_inv);
    }
    if (biased) {
      const float* bias = &sB[buf][wave / RW][BM - 1 + h * 4 - my_row];
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < 16; ++i) s2[c][i] += bias[c * 32 + (i / 4) * 8 + i % 4];
    }
    const bool masked = key0 + BN - 1 > p0 + row0 || a.window > 0 || a.chunk > 0;
    if (masked) {
      const int upto = pos_row - key0 - h * 4, from = lo_row - key0 - h * 4;
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = c * 32 + (i / 4) * 8 + i % 4;
          const bool vis = (key <= upto) & (key > from);
          s2[c][i] = vis ? s2[c][i] : -INFINITY;
        }
    }
    if (BIAS || masked) mx = largest(s2);
  };
  const int j16 = lane % 16, dsub = (lane / 16) % 2;
  int v_at[ND];
#pragma unroll
  for (int t = 0; t < ND; ++t)
    v_at[t] = (h * 4 + j16 / 4) * HD * 2 + (((t * 4 + dsub * 2 + (j16 % 4) / 2) ^ value_swizzle<HD>(j16 / 4)) << 4) + 8 * (j16 % 2);
  // O^T += V^T P^T
  auto values = [&](const bf16* sV, const bf16x8 (&pf)[4]) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int t = 0; t < ND; ++t) {
        const short4v v0 = lds_read_transposed(sV, v_at[t] + kk * 32 * HD);
        const short4v v1 = lds_read_transposed(sV, v_at[t] + (kk * 32 + 16) * HD);
        const short8v both = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, both), pf[kk], o[t], 0, 0, 0);
      }
  };
  floatx16 s_a[2], s_b[2];
  float mx;                    // this lane's largest of the tile's raw scores
  bf16x8 p_a[4], p_b[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) p_b[kk] = zero8;
  const int kt_last = kt_stop - 1;
  // Tile kt: its weights, the scores of tile kt + 1 and the values of tile kt - 1, side by side.
  auto step = [&](int kt, bf16* sK, const bf16* sKn, bf16* sV, const bf16* sVp, int buf, floatx16 (&s_cur)[2], floatx16 (&s_next)[2],
                  bf16x8 (&p_cur)[4], bf16x8 (&p_prev)[4]) {
    if (min(kt + 2, kt_last) - ids_from >= WAVE) load_ids(kt);
    if (biased) {
      put_bias(1 - buf);
      ask_bias(kt + 2);
    }
    bring(kpages, false, sK, min(kt + 2, kt_last));
    if (kt > kt_first) bring(vpages, true, sV, kt);      // (the first one's were asked for with the first keys)
    shape(buf, s_cur, kt * BN, mx);
    mx = halves_max(mx);
    const float m_new = fmaxf(m, mx);
    const float keep = __builtin_amdgcn_exp2f((m - m_new) * scale2);
    const float shift = -m_new * scale2;
    m = m_new;
    l *= keep;
    // One matrix instruction at a time with a share of the vector instructions behind it (32 to 40 cycles of each), in this order: a wave
    // issues in order, and a block of either would leave the other's units idle.
    constexpr int NQ = 2 * DS, ALL = NQ + 4 * ND, AHEAD = 3, PAIRS = 16, EVERY = ALL / PAIRS;
    bf16x8 frag[AHEAD + 1];
    float x[PAIRS][2];
    auto fetch = [&](int j) {
      if (j < NQ) {
        frag[j % (AHEAD + 1)] = *(const bf16x8*)((const char*)sKn + k_at[j / 2] + (j % 2) * 64 * HD);
      } else {
        const int kk = (j - NQ) / ND, t = (j - NQ) % ND;
        const short4v v0 = lds_read_transposed(sVp, v_at[t] + kk * 32 * HD);
        const short4v v1 = lds_read_transposed(sVp, v_at[t] + (kk * 32 + 16) * HD);
        frag[j % (AHEAD + 1)] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    };
    auto score = [&](int e) -> float& { return x[e / 2][e % 2]; };
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) fetch(j);
    score(0) = fmaf(s_cur[0][0], scale2, shift);
    score(1) = fmaf(s_cur[0][1], scale2, shift);
    __builtin_amdgcn_sched_barrier(0);
    float mxn = 0.f;
#pragma unroll
    for (int j = 0; j < ALL; ++j) {
      if (j >= 2 && j - 2 < NQ) HOLD(s_next[j % 2]);
      if (j - 2 >= NQ) HOLD(o[(j - 2 - NQ) % ND]);
      if (j < NQ) {
        const int c = j % 2;
        if (j < 2) {
#pragma unroll
          for (int i = 0; i < 16; ++i) s_next[c][i] = 0.f;
        }
        s_next[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag[j % (AHEAD + 1)], qf[j / 2], s_next[c], 0, 0, 0);
      } else {
        const int kk = (j - NQ) / ND, t = (j - NQ) % ND;
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag[j % (AHEAD + 1)], p_prev[kk], o[t], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (j + AHEAD < ALL) fetch(j + AHEAD);
      if (j % EVERY == 0) {
        const int u = j / EVERY;      // this pair's exponentials, the next one's arguments, the sum and the rounding of the one before
        if (u + 1 < PAIRS) {
          score(2 * u + 2) = fmaf(s_cur[(2 * u + 2) / 16][(2 * u + 2) % 16], scale2, shift);
          score(2 * u + 3) = fmaf(s_cur[(2 * u + 3) / 16][(2 * u + 3) % 16], scale2, shift);
        }
        score(2 * u) = __builtin_amdgcn_exp2f(score(2 * u));
        score(2 * u + 1) = __builtin_amdgcn_exp2f(score(2 * u + 1));
        HOLD(score(2 * u));
        HOLD(score(2 * u + 1));
        if (u + 1 < PAIRS) {
          HOLD(score(2 * u + 2));
          HOLD(score(2 * u + 3));
        }
        if (u > 0) {
          l += score(2 * u - 2);
          l += score(2 * u - 1);
          p_cur[(u - 1) / 4][(2 * u - 2) % 8] = (bf16)score(2 * u - 2);
          p_cur[(u - 1) / 4][(2 * u - 1) % 8] = (bf16)score(2 * u - 1);
          HOLD(l);
          if (u % 4 == 0) HOLD(p_cur[u / 4 - 1]);
        }
      }
      if (!BIAS && j == NQ + 1) mxn = fmaxf(s_next[0][0], s_next[1][15]);
      if (!BIAS && j > NQ) {      // the next scores' largest
        constexpr int SHARE = (15 + ALL - NQ - 2) / (ALL - NQ - 1);
#pragma unroll
        for (int n = (j - NQ - 1) * SHARE; n < (j - NQ) * SHARE && n < 15; ++n) {
          const int i = 2 * n + 1;
          mxn = fmaxf(fmaxf(mxn, s_next[i / 16][i % 16]), s_next[(i + 1) / 16][(i + 1) % 16]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    l += score(2 * PAIRS - 2);
    l += score(2 * PAIRS - 1);
    p_cur[3][6] = (bf16)score(2 * PAIRS - 2);
    p_cur[3][7] = (bf16)score(2 * PAIRS - 1);
    HOLD(p_cur[3]);
    mx = mxn;
    if (__builtin_amdgcn_ballot_w64(keep != 1.f) != 0) {
#pragma unroll
      for (int t = 0; t < ND; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[t][i] *= keep;
    }
    // this wave's part of the next step's tiles has landed and its reads of LDS are through (the barrier covers the other waves')
    barrier_behind_loads<0>();
  };
  if (kt_first == kt_last) {
    // one tile: nothing to run side by side (45 rows of 16 heads 5.9 us a call, through the steps below 6.8)
    load_ids(kt_first);
    if (biased) ask_bias(kt_first);
    bring(kpages, false, sK0, kt_first);
    bring(vpages, true, sV0, kt_first);
    if (biased) put_bias(0);
    __syncthreads();
    scores(sK0, s_a);
    clear_tail(sV0, kt_first);
    shape(0, s_a, kt_first * BN, mx);
    if (!BIAS) mx = largest(s_a);
    m = fmaxf(m, halves_max(mx));
    const float shift = -m * scale2;
#pragma unroll
    for (int e = 0; e < 32; ++e) {
      const float p = __builtin_amdgcn_exp2f(fmaf(s_a[e / 16][e % 16], scale2, shift));
      l += p;
      p_a[e / 8][e % 8] = (bf16)p;
    }
    values(sV0, p_a);
  } else if (kt_first < kt_stop) {
    load_ids(kt_first);
    if (biased) ask_bias(kt_first);
    bring(kpages, false, sK0, kt_first);
    bring(vpages, true, sV0, kt_first);
    bring(kpages, false, sK1, kt_first + 1);
    for (int c = tid; c < BN * CPR; c += NT) *(uint4*)&sV1[c * 8] = make_uint4(0, 0, 0, 0);   // (the values of no tile, with weights of zero)
    if (biased) {
      put_bias(0);
      ask_bias(kt_first + 1);
    }
    __syncthreads();
    scores(sK0, s_a);
    mx = largest(s_a);
    __syncthreads();
    int kt = kt_first;
    for (; kt + 1 < kt_stop; kt += 2) {
      step(kt, sK0, sK1, sV0, sV1, 0, s_a, s_b, p_a, p_b);
      step(kt + 1, sK1, sK0, sV1, sV0, 1, s_b, s_a, p_b, p_a);
    }
    if (kt < kt_stop) {
      step(kt, sK0, sK1, sV0, sV1, 0, s_a, s_b, p_a, p_b);
      clear_tail(sV0, kt_last);
      values(sV0, p_a);
    } else {
      clear_tail(sV1, kt_last);
      values(sV1, p_b);
    }
  }

  // A weight of zero makes a value that is not finite a NaN, in rows of the wave that do not see its key too.  Rows that come out
  // so are taken again, a row at a time over its own keys: scores with a key a lane, sums with a place or two of the head a lane.
  // (The look at the results, us, 32 heads of 64: 512 rows 11.50 -> 11.55, 2,048 35.9 / 35.8, calls of 5 us 0.1 to 0.2 more.)
  float probe = 0.f;
#pragma unroll
  for (int t = 0; t < ND; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) probe = fmaf(o[t][i], 0.f, probe);
  const uint64_t spoilt = __builtin_amdgcn_ballot_w64(row0 + lr < rows_here && !(probe == 0.f) && l < INFINITY);   // (a sum that is none: every place is)
  if (__builtin_expect(spoilt != 0, 0)) {
    auto offset_of = [&](int key) {
      const int page = table[key >> a.page_shift];
      return (size_t)min(max(page, 0), a.num_pages - 1) * page_stride + head_off + (size_t)(key & (a.page_size - 1)) * HD;
    };
#pragma unroll 1
    for (uint32_t rows = (uint32_t)spoilt | (uint32_t)(spoilt >> 32); rows != 0; rows &= rows - 1) {
      const int n = __builtin_ctz(rows), upto = __builtin_amdgcn_readlane(pos_row, n), from = __builtin_amdgcn_readlane(lo_row, n);
      const float shift = -__uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(m), n)) * scale2;
      const bf16* qr = q + (size_t)(n0 + row0 + n) * a.ldq + (size_t)head * HD;
      float sum[HD / WAVE] = {};
#pragma unroll 1
      for (int key0 = max(kt_first, (from + 1) / BN) * BN; key0 <= min(upto, kt_stop * BN - 1); key0 += BN) {
        const int key = min(key0 + lane, last_pos);
        const bf16* kr = kpages + offset_of(key);
        float s = 0.f;
#pragma unroll 1
        for (int d = 0; d < HD; ++d) s = fmaf(to_float(kr[d]), to_float(qr[d]), s);
        if constexpr (CAP) s = cap_raw * tanhf(s * cap_inv);
        if (biased) s += a.bias[(size_t)head * a.bias_len + min(max(upto - key, 0), a.bias_len - 1)];
        const float p = to_float((bf16)__builtin_amdgcn_exp2f(fmaf(s, scale2, shift)));
#pragma unroll 1
        for (int j = max(0, from + 1 - key0); j < BN && key0 + j <= upto; ++j) {
          const bf16* vr = vpages + offset_of(key0 + j);
          const float w = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(p), j));
#pragma unroll
          for (int t = 0; t < HD / WAVE; ++t) sum[t] = fmaf(w, to_float(vr[t * WAVE + lane]), sum[t]);
        }
      }
#pragma unroll
      for (int t = 0; t < ND; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float v = __shfl(sum[t * 32 / WAVE], (t * 32 + (i / 4) * 8 + h * 4 + i % 4) % WAVE, WAVE);
          if (lr == n) o[t][i] = v;
        }
    }
  }

  l = halves_sum(l);
  const int row = row0 + lr;
  if (row >= rows_here) return;
  if (a.n_splits > 1) {
    float* ps = partial + (((size_t)(n0 + row) * a.nh + head) * a.n_splits + blockIdx.z) * (HD + 2);
    if (h == 0) {
      ps[0] = m * a.scale;
      ps[1] = l;
    }
#pragma unroll
    for (int t = 0; t < ND; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) ps[2 + t * 32 + (i / 4) * 8 + h * 4 + i % 4] = o[t][i];
    return;
  }
  if (a.sink) l += __expf(a.sink[head] - m * a.scale);
  const float inv = 1.0f / l;
  bf16* dst = out + (size_t)(n0 + row) * a.ldo + (size_t)head * HD + h * 4;
#pragma unroll
  for (int t = 0; t < ND; ++t)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const bf16x4 v = {(bf16)(o[t][b * 4] * inv), (bf16)(o[t][b * 4 + 1] * inv), (bf16)(o[t][b * 4 + 2] * inv), (bf16)(o[t][b * 4 + 3] * inv)};
      if (a.ldo % 4 == 0) {
        *(bf16x4*)(dst + t * 32 + b * 8) = v;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) dst[t * 32 + b * 8 + i] = v[i];
      }
    }
}

template <int HD, int HW>
void launch_heads(const bf16* q, const bf16* k, const bf16* v, bf16* out, float* partial, const PrefillArgs& a, int n_rows, hipStream_t stream) {
  constexpr int RW = 4 / HW;
  const dim3 grid((ceil_div(n_rows, 32 * RW) + a.n_req) * (a.nh / HW), 1, a.n_splits);
  if (a.softcap > 0.f) attention_prompt_kernel<HD, HW, RW, SCORES_CAPPED><<<grid, 256, 0, stream>>>(q, k, v, out, partial, a);
  else if (a.bias) attention_prompt_kernel<HD, HW, RW, SCORES_BIASED><<<grid, 256, 0, stream>>>(q, k, v, out, partial, a);
  else attention_prompt_kernel<HD, HW, RW, SCORES_PLAIN><<<grid, 256, 0, stream>>>(q, k, v, out, partial, a);
}
template <int HD>
void launch_head_size(const bf16* q, const bf16* k, const bf16* v, bf16* out, float* partial, const PrefillArgs& a, int n_rows, hipStream_t stream) {
  const int group = a.nh / a.nkv;
  if (group % 4 == 0) launch_heads<HD, 4>(q, k, v, out, partial, a, n_rows, stream);
  else if (group % 2 == 0) launch_heads<HD, 2>(q, k, v, out, partial, a, n_rows, stream);
  else launch_heads<HD, 1>(q, k, v, out, partial, a, n_rows, stream);
}
}  // namespace

void launch_prompt_attention(const bf16* q, const bf16* kpages, const bf16* vpages, bf16* out, float* partial, const PrefillArgs& a,
                             int n_rows, hipStream_t stream) {
  if (a.hd == 64) launch_head_size<64>(q, kpages, vpages, out, partial, a, n_rows, stream);
  else launch_head_size<128>(q, kpages, vpages, out, partial, a, n_rows, stream);
}
