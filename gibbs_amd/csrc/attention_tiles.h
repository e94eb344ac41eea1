// Paged decode attention for the shapes that models bring: heads of 64 or 128, 1, 2, 4 or 8 query heads to a kv head, pages of
// 16 keys or a larger power of two, and (raw rows) no rotation or one of whole heads by halves.  attention_decode.h has what
// both kernels compute, the merge of the slices and the kernel for every other shape.
//
// What a call costs at few rows is not its bytes (33 MB at 8 rows of 2,100 keys are 5 us, it took 16.5) but the length of the
// path: an instruction of a wave takes 2 ns, a dependent access of memory 0.3 to 0.8 us, and the general kernel is 5,700
// instructions long, with a branch for each element that may lie outside a head.  Here sizes are known when the kernel is
// compiled, and
//   * where a row's keys are whole and in one slice, a wave knows its page ids' places without the row's position: ids and position
//     are asked for together, the keys next;
//   * a page id holds for 16 keys, so it is a scalar: the keys' and values' addresses are a scalar base and the lane's 16 bytes;
//   * every wave prepares all query heads (and the row's own key) at once, a head to each group of lanes, instead of a head a
//     wave: the queries reach the matrix operand by lane permutes, no LDS and no barrier in front of the walk;
//   * the waves' results are folded, and the slices merged, by all threads, two elements each.
// Which keys a slice and a wave take, and the order in which their results are folded, are the general kernel's: the bits of a row are the same
// in both.  (Where the row's first key lies inside a tile, as a window has it, the tiles begin in front of it, at a multiple of 32, and
// the bits are others.)
//
// Measured (us a call in a captured chain of calls over caches of their own, the general kernel -> this one, both in the slices of 4 waves that
// decode_splits gives): 16 query heads of 64 in 8 groups, 1 row of 40 keys 7.7 -> 4.4, of 500 11.1 -> 6.9; 32 heads in 8, 1 row of 2,100 12.5 -> 8.2, of
// 16,000 21.0 -> 20.0 (64 slices, whose merge is 6); 8 rows of 2,100 17.2 -> 12.6 (33 MB: 5.3 at the rate of a kernel that only reads); 64 rows of 1,000
// 34.8 -> 28.8 (131 MB: 21); 8 rows of 520 with a bias 11.8 -> 7.9, with a sink 10.6 -> 7.3; 16 heads of 128 in 4, 8 rows of 520 13.8 -> 8.4.
#pragma once

namespace {
struct TilesArgs {
  bf16* vpages;
  bf16* out;
  float* partial;
  long ldo;
  int num_pages, nh, nkv;
  uint32_t per_tile;      // 2^32 over the waves of all slices, rounded up
  float scale;
  int merge_here;
  // raw rows
  const float* q_gain;    // [HD], or null with k_gain
  const float* k_gain;
  float eps;
  const float* inv_freq;  // [HD / 2] or null
  const float2* cs_table; // [table_len, HD / 2]
  int table_len;
  // prepared rows
  const float* bias;      // [nh, bias_len], or null
  int bias_len;
  const float* sink;      // [nh], or null
  float softcap;
  int window, chunk;      // > 0: a row sees its last `window` keys, or those of its own stretch of `chunk` positions
};

__device__ __forceinline__ unsigned long long load_through2(const float* p) {
  return __hip_atomic_load((const unsigned long long*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float low_half(unsigned long long v) { return __uint_as_float((uint32_t)v); }
__device__ __forceinline__ float high_half(unsigned long long v) { return __uint_as_float((uint32_t)(v >> 32)); }

// What the first loads hang on are scalar arguments: those arrive in registers with the wave, the struct by loads.
// packed: slices << 8 | rows have a map to requests << 7 | a window or chunks << 6 | log2(keys of a page).
// EXTRA: prepared rows with a bias, a sink or capped scores (a kernel of its own: the others walk without their code).
template <int HD, int GT, bool RAW, int NW, bool EXTRA>
__global__ __launch_bounds__(NW * WAVE, HD == 64 ? 4 : 2) void attention_tiles_kernel(
    const int* __restrict__ pos_, const int* __restrict__ table_, const int* __restrict__ row_req, bf16* __restrict__ kpages,
    const bf16* __restrict__ q_, int ldq, int max_pages, uint32_t page_bytes, uint32_t packed, TilesArgs a) {
  constexpr int LPK = HD / EPL, KPW = WAVE / LPK;      // lanes of a key, keys of a load instruction
  constexpr int LPT = TILE / KPW, LPH = LPT / 2;       // load instructions of a tile, of 16 keys
  constexpr int LDT = HD + 8;                          // row of a tile in LDS (padded against bank conflicts)
  constexpr int DT = HD / 16, DS = HD / 32;
  constexpr int WAVE_LDS = 2 * TILE * LDT;
  static_assert(GT * HD * 4 <= WAVE_LDS * 2, "a wave's results take the place of its tiles");
  __shared__ __attribute__((aligned(16))) bf16 s_tiles[NW * WAVE_LDS];
  __shared__ float s_ml[NW][GT][2];
  __shared__ int s_last;

  const int row = blockIdx.x, kvh = blockIdx.y, split = blockIdx.z;
  const int p = pos_[row];
  __builtin_amdgcn_sched_barrier(0);                   // (asked for first)
  const int page_shift = packed & 63, n_splits = packed >> 8;
  const uint32_t per_tile = a.per_tile;
  const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int grp = lane / LPK, sub = lane % LPK, e0 = sub * EPL;
  const int lr = lane % 16, g4 = lane / 16;
  int req = row;
  if (packed & 128) {
    req = row_req[row];
    asm volatile("" : "+s"(req));                      // (waited for here, so that a step without a map waits for nothing)
  }
  const int* table = table_ + (size_t)req * max_pages;
  // the first key that the row sees, and the tile it lies in; the wave's tiles: first, first + NW, ... (0 and the wave without waiting for the
  // position, where a row's keys are whole and in one slice)
  int lo = 0, base = 0, first = wave, per_slice = 0;
  if (packed & 64) {
    lo = !RAW && a.chunk > 0 ? p - p % a.chunk : max(0, p - a.window + 1);
    base = lo / TILE * TILE;
  }
  if (n_splits > 1) {
    // ceil(tiles / (slices NW)) to each wave: a product in place of the division, at most one too many
    const uint32_t waves = n_splits * NW, x = (uint32_t)max(0, p - base + TILE) / TILE + waves - 1;
    uint32_t rounds = __umulhi(x, per_tile);
    if (rounds * waves > x) --rounds;
    per_slice = rounds * NW;
    first = split * per_slice + wave;
  }
  // lane l of the wave holds the page id of 16 keys: half l % 2 of its tile l / 2 (of 32 tiles at a time)
  auto ask_ids = [&](int round) {
    const int key = base + (first + (round * 32 + lane / 2) * NW) * TILE + 16 * (lane % 2);
    return table[min(key >> page_shift, max_pages - 1)];
  };
  int ids = ask_ids(0);
  __builtin_amdgcn_sched_barrier(0);                   // (nothing that hangs on the struct of arguments stands in front of this load)

  // the queries, and what prepares them, while ids and position are on their way
  constexpr int GPW = WAVE / LPK;                      // vectors (heads) that a wave holds at a time
  constexpr int PASSES = (GT + GPW) / GPW;             // the query heads and the row's own key
  uint4 raw[RAW ? PASSES : 1];
  uint4 v_new = make_uint4(0, 0, 0, 0);
  float gain[RAW ? PASSES : 1][EPL];
  bf16x8 qb[DS];
  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  const bf16* qrow = q_ + (size_t)row * ldq;
  if constexpr (RAW) {
#pragma unroll
    for (int j = 0; j < PASSES; ++j) {
      const int v = j * GPW + grp;                     // < GT: a query head; GT: the key
      const int head = v < GT ? kvh * GT + v : a.nh + kvh;
      raw[j] = *(const uint4*)(qrow + head * HD + e0);
      if (a.q_gain) {
        const float* gp = (v < GT ? a.q_gain : a.k_gain) + e0;
        const floatx4 g0 = *(const floatx4*)gp, g1 = *(const floatx4*)(gp + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) { gain[j][i] = g0[i]; gain[j][4 + i] = g1[i]; }
      }
    }
    v_new = *(const uint4*)(qrow + (a.nh + a.nkv + kvh) * HD + e0);
  } else {
    // B operands of S^T = K Q^T: column lr is query head lr, d = s*32 + g4*8 .. +8
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      const bf16x8 q8 = *(const bf16x8*)(qrow + (kvh * GT + min(lr, GT - 1)) * HD + s * 32 + g4 * 8);
      qb[s] = lr < GT ? q8 : zero8;
    }
  }

  const int all_tiles = (p - base + TILE) / TILE;
  const int n_tiles = n_splits > 1 ? min(all_tiles, (split + 1) * per_slice) : all_tiles;      // where the slice ends
  const int kv_bytes = kvh << page_shift;              // keys of a page in front of this head's (times HD * 2 bytes)
  uint4 kreg[LPT], vreg[LPT];
  float bnext[EXTRA ? 8 : 1];
  const float* bias = EXTRA && a.bias ? a.bias + (size_t)(kvh * GT + min(lr, GT - 1)) * a.bias_len : nullptr;
  auto fetch = [&](int tile, int j) {                  // tile j of the wave (of the 32 whose ids it holds)
    const int key = base + tile * TILE;
    if (EXTRA && bias) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) bnext[c * 4 + i] = bias[min(max(p - (key + c * 16 + g4 * 4 + i), 0), a.bias_len - 1)];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t id = min(max(__builtin_amdgcn_readlane(ids, 2 * j + h), 0), a.num_pages - 1);   // never read outside the pool
      const int within = (key + 16 * h) & ((1 << page_shift) - 1);
      const size_t off = (size_t)id * page_bytes + (size_t)(uint32_t)(kv_bytes + within) * (HD * 2);
      const char* kb = (const char*)kpages + off;
      const char* vb = (const char*)a.vpages + off;
#pragma unroll
      for (int i = 0; i < LPH; ++i) {
        kreg[h * LPH + i] = *(const uint4*)(kb + lane * 16 + i * 1024);
        vreg[h * LPH + i] = *(const uint4*)(vb + lane * 16 + i * 1024);
      }
    }
  };
  if (first < n_tiles) fetch(first, 0);
  __builtin_amdgcn_sched_barrier(0);                   // the keys are asked for before the queries are prepared

  uint4 k_new = make_uint4(0, 0, 0, 0);
  constexpr int KEY_PASS = GT / GPW, KEY_GRP = GT % GPW;
  if constexpr (RAW) {
    constexpr int half = HD / 2;
    float c8[EPL], s8[EPL];
    const bool rotate = a.inv_freq != nullptr;
    if (rotate) {
      if (p < a.table_len) {
        const float2* cs = a.cs_table + (size_t)p * half + (e0 & (half - 1));
#pragma unroll
        for (int i = 0; i < EPL; i += 2) {
          const floatx4 t = *(const floatx4*)(cs + i);
          c8[i] = t[0]; s8[i] = t[1]; c8[i + 1] = t[2]; s8[i + 1] = t[3];
        }
      } else {                                         // beyond the table: one element at a time, the code is long
#pragma unroll 1
        for (int i = 0; i < EPL; ++i) {
          float c, s;
          rope_cos_sin((float)p * a.inv_freq[(e0 + i) & (half - 1)], &c, &s);
#pragma unroll
          for (int k = 0; k < EPL; ++k) {
            c8[k] = k == i ? c : c8[k];
            s8[k] = k == i ? s : s8[k];
          }
        }
      }
    }
    uint4 ready[PASSES];
#pragma unroll
    for (int j = 0; j < PASSES; ++j) {
      float v[EPL];
      unpack8(raw[j], v);
      if (a.q_gain) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < EPL; ++i) ss += v[i] * v[i];
        ss = group_sum<LPK>(ss);
        const float sc = 1.0f / sqrtf(ss / (float)HD + a.eps);
#pragma unroll
        for (int i = 0; i < EPL; ++i) v[i] = v[i] * sc * gain[j][i];
      }
      if (rotate) {
        const bool low = e0 < half;
#pragma unroll
        for (int i = 0; i < EPL; ++i) {
          const float other = lane_xor<LPK / 2>(v[i]);
          v[i] = fmaf(v[i], c8[i], low ? -(other * s8[i]) : other * s8[i]);   // (the product that is rounded is the one the compiler rounds in norm_rope8)
        }
      }
      ready[j] = pack8(v);                             // bfloat16, as the pages hold keys and other kernels queries
    }
    k_new = ready[KEY_PASS];                           // (valid in the lanes of group KEY_GRP)
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      const int src = ((lr % GPW) * LPK + s * 4 + g4) * 4;
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t mine[4] = {ready[0].x, ready[0].y, ready[0].z, ready[0].w};
        w[i] = __builtin_amdgcn_ds_bpermute(src, mine[i]);
        if constexpr (GT > GPW) {
          const uint32_t mine1[4] = {ready[1].x, ready[1].y, ready[1].z, ready[1].w};
          const uint32_t w1 = __builtin_amdgcn_ds_bpermute(src, mine1[i]);
          w[i] = lr < GPW ? w[i] : w1;
        }
        w[i] = lr < GT ? w[i] : 0u;
      }
      typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
      qb[s] = __builtin_bit_cast(bf16x8, uint4v{w[0], w[1], w[2], w[3]});
    }
  }

  // the walk: this lane holds, of query head lr, the scores of 8 keys per tile, and of the output the elements
  // d = t*16 + g4*4 + i.  A tile travels memory -> registers (one tile ahead) -> the wave's own patch of LDS
  // (no barrier: only this wave reads it) -> matrix instructions.
  float mm_m = -1e30f, mm_l = 0.f;   // (a finite stand-in for 'no key yet': exp2 of anything minus it is 0)
  floatx4 mm_o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) mm_o[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  bf16 (*tK)[LDT] = reinterpret_cast<bf16 (*)[LDT]>(s_tiles + (size_t)wave * WAVE_LDS);
  bf16 (*tV)[LDT] = tK + TILE;
  const float scale2 = a.scale * 1.44269504088896340736f;
  int j = 0, round = 0;
  for (int tile = first; tile < n_tiles; tile += NW) {
    const int t0 = base + tile * TILE;
    // (what lies in a page outside the keys that the row sees may be anything: 0 times it need not be 0.  The row's own
    // key and value come from the registers)
    const int end = RAW ? p : p + 1;
    if (t0 + TILE > end || t0 < lo) {
#pragma unroll
      for (int i = 0; i < LPT; ++i) {
        const int key = t0 + i * KPW + grp;
        if (key >= end || key < lo) kreg[i] = vreg[i] = make_uint4(0, 0, 0, 0);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the reads of the previous tile are through
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      *(uint4*)&tK[i * KPW + grp][e0] = kreg[i];
      *(uint4*)&tV[i * KPW + grp][e0] = vreg[i];
    }
    float b8[EXTRA ? 8 : 1];
    if (EXTRA) {
#pragma unroll
      for (int i = 0; i < 8; ++i) b8[i] = bnext[i];
    }
    if (tile + NW < n_tiles) {
      if (++j == 32) {
        j = 0;
        ids = ask_ids(++round);
      }
      fetch(tile + NW, j);
    }
    __builtin_amdgcn_sched_barrier(0);  // the loads above stay ahead of the arithmetic below
    if (RAW && t0 + TILE > p) {   // the wave's last tile: the row's own key and value, here and in their page
      const int id = __builtin_amdgcn_readlane(ids, 2 * j + (p - t0) / 16);
      if (grp == KEY_GRP) {
        *(uint4*)&tK[p - t0][e0] = k_new;
        *(uint4*)&tV[p - t0][e0] = v_new;
        if (id >= 0 && id < a.num_pages && (p >> page_shift) < max_pages) {   // the host never asks for another; never write outside
          const size_t off = (size_t)id * page_bytes + (size_t)(uint32_t)(kv_bytes + (p & ((1 << page_shift) - 1))) * (HD * 2) + e0 * 2;
          *(uint4*)((char*)kpages + off) = k_new;
          *(uint4*)((char*)a.vpages + off) = v_new;
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the tile is in LDS
    floatx4 s4[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      s4[c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < DS; ++s)
        s4[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)&tK[c * 16 + lr][s * 32 + g4 * 8], qb[s], s4[c], 0, 0, 0);
    }
    if (EXTRA && a.softcap > 0.f) {   // (in the raw scores' units: the scale follows)
      const float cap_raw = a.softcap / a.scale, cap_inv = a.scale / a.softcap;
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) s4[c][i] = cap_raw * tanhf(s4[c][i] * cap_inv);
    }
    if (EXTRA && bias) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) s4[c][i] += b8[c * 4 + i];
    }
    // keys that the row does not see (in the first tile and the last); maximum of the raw scores (the scale is positive)
    if (t0 + TILE > p + 1 || t0 < lo) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = t0 + c * 16 + g4 * 4 + i;
          s4[c][i] = key <= p && key >= lo ? s4[c][i] : -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s4[c][i]);
    mx = row4_max(mx);
    const float m_new = fmaxf(mm_m, mx);
    const float keep = __builtin_amdgcn_exp2f((mm_m - m_new) * scale2);
    const float shift = -m_new * scale2;
    mm_m = m_new;
    mm_l *= keep;
    bf16x8 pf;   // P^T as the B operand: element e is key (e / 4) * 16 + g4 * 4 + e % 4 of the tile
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float pr = __builtin_amdgcn_exp2f(fmaf(s4[c][i], scale2, shift));
        mm_l += pr;
        pf[c * 4 + i] = (bf16)pr;
      }
#pragma unroll
    for (int t = 0; t < DT; ++t) {
#pragma unroll
      for (int i = 0; i < 4; ++i) mm_o[t][i] *= keep;
      // V^T of d = t*16 + lr, the same 8 keys: two transposing reads of 4 keys each
      const short4v v0 = lds_read_transposed(&tV[g4 * 4 + lr / 4][t * 16 + 4 * (lr % 4)]);
      const short4v v1 = lds_read_transposed(&tV[16 + g4 * 4 + lr / 4][t * 16 + 4 * (lr % 4)]);
      typedef short short8v __attribute__((ext_vector_type(8)));
      const short8v both = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
      mm_o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, both), pf, mm_o[t], 0, 0, 0);
    }
  }

  // the waves' results take the place of their tiles (the wave's own patch: its reads are through), then all threads fold them
  float* mine = reinterpret_cast<float*>(s_tiles + (size_t)wave * WAVE_LDS);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  const float total = row4_sum(mm_l);
  if (lr < GT) {
    if (g4 == 0) { s_ml[wave][lr][0] = mm_m * a.scale; s_ml[wave][lr][1] = total; }
#pragma unroll
    for (int t = 0; t < DT; ++t) *(floatx4*)(mine + lr * HD + t * 16 + g4 * 4) = mm_o[t];
  }
  __syncthreads();
  constexpr int PAIRS = GT * HD / 2;
  const bool merge_here = n_splits > 1 && a.merge_here;
  float* const row_partial = a.partial + ((size_t)row * a.nh + kvh * GT) * n_splits * (HD + 2);
  bf16* const row_out = a.out + (size_t)row * a.ldo + kvh * GT * HD;
  auto put = [&](int g, int e, float L, float v0, float v1) {
    const float inv = 1.0f / L;
    typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
    *(bf16x2*)(row_out + g * HD + e) = bf16x2{(bf16)(v0 * inv), (bf16)(v1 * inv)};
  };
#pragma unroll
  for (int i0 = 0; i0 < PAIRS; i0 += NW * WAVE) {
    const int i = i0 + threadIdx.x;
    if (PAIRS % (NW * WAVE) != 0 && i >= PAIRS) break;
    const int g = i / (HD / 2), e = i % (HD / 2) * 2;
    auto values = [&](int w) { return *(const float2*)(reinterpret_cast<const float*>(s_tiles + (size_t)w * WAVE_LDS) + g * HD + e); };
    float M = s_ml[0][g][0], L = s_ml[0][g][1], v[2] = {values(0).x, values(0).y};
#pragma unroll
    for (int w = 1; w < NW; ++w) {
      const float2 x = values(w);
      const float more[2] = {x.x, x.y};
      fold<2>(M, L, v, s_ml[w][g][0], s_ml[w][g][1], more);
    }
    if (n_splits == 1) {
      if (EXTRA && a.sink) L += __expf(a.sink[kvh * GT + g] - M);
      put(g, e, L, v[0], v[1]);
    } else {
      float* ps = row_partial + ((size_t)g * n_splits + split) * (HD + 2);
      if (merge_here) {
        // another workgroup, on another L2, reads them in this same kernel: written through
        if (e == 0) store_through2(ps, M, L);
        store_through2(ps + 2 + e, v[0], v[1]);
      } else {
        if (e == 0) *(float2*)ps = make_float2(M, L);
        *(float2*)(ps + 2 + e) = make_float2(v[0], v[1]);
      }
    }
  }
  if (!merge_here) return;
  // The slice that finishes last merges them all (attention_decode.h: why this takes no fence).
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  int* counter = g_merge_counters + (size_t)row * gridDim.y + blockIdx.y;
  if (threadIdx.x == 0) {
    const int before = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = before == n_splits - 1;
    if (s_last) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next call
  }
  __syncthreads();
  if (!s_last) return;
#pragma unroll 1
  for (int i = threadIdx.x; i < PAIRS; i += NW * WAVE) {
    const int g = i / (HD / 2), e = i % (HD / 2) * 2;
    const float* ps = row_partial + (size_t)g * n_splits * (HD + 2);
    float M = -INFINITY, L = 0.f, v0 = 0.f, v1 = 0.f;
#pragma unroll 1
    for (int s0 = 0; s0 < n_splits; s0 += 8) {       // eight slices' loads in flight at a time
      unsigned long long ml[8], av[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float* sp = ps + (size_t)min(s0 + k, n_splits - 1) * (HD + 2);   // (beyond the last slice: the last one again, weighted 0 below)
        ml[k] = load_through2(sp);
        av[k] = load_through2(sp + 2 + e);
      }
      float Mn = M;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (s0 + k < n_splits) Mn = fmaxf(Mn, low_half(ml[k]));
      const float keep = M == -INFINITY ? 0.f : __expf(M - Mn);
      L *= keep; v0 *= keep; v1 *= keep;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float w = (s0 + k < n_splits && low_half(ml[k]) != -INFINITY) ? __expf(low_half(ml[k]) - Mn) : 0.f;
        L = fmaf(w, high_half(ml[k]), L);
        v0 = fmaf(w, low_half(av[k]), v0);
        v1 = fmaf(w, high_half(av[k]), v1);
      }
      M = Mn;
    }
    if (EXTRA && a.sink) L += __expf(a.sink[kvh * GT + g] - M);   // (a sink counts once, whatever the number of slices)
    put(g, e, L, v0, v1);
  }
}

// What the kernel takes; the rest goes to the general one.
template <bool RAW>
bool tiles_take(const DecodeArgs& a, int kind, const bf16* q, const bf16* kpages, const bf16* vpages, const bf16* out, const float* partial) {
  const int G = a.nh / a.nkv;
  auto at = [](const void* p, int bytes) { return (uintptr_t)p % bytes == 0; };
  if (kind == 1 || (a.hd != 64 && a.hd != 128) || (G != 1 && G != 2 && G != 4 && G != 8) || a.nkv > 65535) return false;
  if (a.page_shift < 4 || (long)a.nkv * a.page_size * a.hd * 2 > 0x7fffffffl) return false;
  if (a.ldq > 0x7fffffffl / 2 || !at(q, 16) || a.ldq % 8 != 0 || !at(kpages, 16) || !at(vpages, 16) || !at(out, 4) || a.ldo % 2 != 0) return false;
  if (a.n_splits > 1 && !at(partial, 8)) return false;
  if (RAW) {
    if (a.inv_freq && !(a.variant == 0 && a.rot == a.hd && a.cs_table && at(a.cs_table, 16))) return false;
    if ((a.q_gain != nullptr) != (a.k_gain != nullptr) || !at(a.q_gain, 16) || !at(a.k_gain, 16)) return false;
  }
  return true;
}

template <int HD, bool RAW, int NW, bool EXTRA>
void launch_tiles(int G, dim3 grid, hipStream_t s, const bf16* q, bf16* k, const DecodeArgs& d, TilesArgs a) {
  const uint64_t waves = (uint64_t)d.n_splits * NW;
  a.per_tile = (uint32_t)(((1ull << 32) + waves - 1) / waves);
  const uint32_t page_bytes = (uint32_t)d.nkv * d.page_size * HD * 2;
  const uint32_t packed = (uint32_t)d.n_splits << 8 | (d.row_req ? 128u : 0u) | (d.window > 0 || d.chunk > 0 ? 64u : 0u) | (uint32_t)d.page_shift;
#define GIBBS_TILES(GT) attention_tiles_kernel<HD, GT, RAW, NW, EXTRA><<<grid, NW * WAVE, 0, s>>>(d.pos, d.table, d.row_req, k, q, (int)d.ldq, d.max_pages, page_bytes, packed, a)
  switch (G) {
    case 1: GIBBS_TILES(1); break;
    case 2: GIBBS_TILES(2); break;
    case 4: GIBBS_TILES(4); break;
    default: GIBBS_TILES(8); break;
  }
#undef GIBBS_TILES
}

template <bool RAW>
void run_tiles(const DecodeArgs& d, int n_rows, int waves, hipStream_t s, const bf16* q, bf16* k, bf16* v, bf16* out, float* partial) {
  TilesArgs a{};
  a.vpages = v; a.out = out; a.partial = partial; a.ldo = d.ldo;
  a.num_pages = d.num_pages; a.nh = d.nh; a.nkv = d.nkv; a.scale = d.scale; a.merge_here = d.merge_here;
  a.q_gain = d.q_gain; a.k_gain = d.k_gain; a.eps = d.eps; a.inv_freq = d.inv_freq; a.cs_table = d.cs_table; a.table_len = d.table_len;
  a.bias = d.bias; a.bias_len = d.bias_len; a.sink = d.sink; a.softcap = d.softcap; a.window = d.window; a.chunk = d.chunk;
  const dim3 grid(n_rows, d.nkv, d.n_splits);
  const int G = d.nh / d.nkv;
  auto go = [&](auto extra) {
    constexpr bool EXTRA = decltype(extra)::value;
    // (heads of 128: 8 waves were no faster anywhere, 8 rows of 2,000 keys in 8 slices 11.7 us and 11.2 with 4)
    if (d.hd == 128) launch_tiles<128, RAW, 4, EXTRA>(G, grid, s, q, k, d, a);
    else if (waves >= 8) launch_tiles<64, RAW, 8, EXTRA>(G, grid, s, q, k, d, a);
    else launch_tiles<64, RAW, 4, EXTRA>(G, grid, s, q, k, d, a);
  };
  if constexpr (!RAW) {
    if (d.bias || d.sink || d.softcap > 0.f) return go(std::true_type{});
  }
  go(std::false_type{});
}
}  // namespace
