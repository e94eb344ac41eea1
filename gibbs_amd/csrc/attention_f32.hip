// Paged causal attention in float32, prompt portions and decoded tokens, on the gfx950 matrix cores: 32-bit operands, products,
// scores, weights and sums throughout (v_mfma_f32_16x16x4_f32), the results of attention_plain.hip to rounding.
//
// A workgroup takes 64 consecutive query rows of one request and one head; 4 waves own 16 of the rows each.  Keys are
// walked in tiles of 64 aligned to absolute key index, K and V as stored ([key][d]) in LDS, the next tile on its way
// in registers and the page ids of the one after it too.  As in the bfloat16 kernel the scores are transposed,
// S^T = K Q^T, so that a lane holds 16 scores of ONE row and its weights are, as they lie, the second operand of
// O^T += V^T P^T.  The contraction may run over d and over the keys in any order: step j of a group of 16 d takes
// d = 4 g + j (g = lane / 16), so that a lane's four steps are one 16-byte read of K, and tile t of O^T takes every
// VEC-th d, so that one read of V serves VEC products.
//
// A wave and tile at head size 64 is 128 matrix instructions of 32 cycles, and about as long again of exponentials and
// of waits that nothing covers: a prompt of some thousand rows has one wave for each SIMD.  16 heads over 8 of the cache, head
// size 64 (in brackets attention_plain.hip, whose lanes read a key each, uncoalesced, and every key once a row): 1,194 rows of a
// prompt 112 us (1,348), 4,096 rows 646 us (11,963; 52 TFLOP/s), 64 rows after 1,000 keys 66 us (518).  Values of twice the
// keys' size (VT): the same walk with V in pieces and pages of its own; 20 rows behind 200 keys, 8 heads over 2 of 64 and 128, 33 us (292 in the plain
// kernel); 8 rows behind 20 9.4 (12.4), 63 8.7 (31); one row behind 7 keys 9.2 (6.9), 20 rows of a prompt 9.4 (11.9): a tile of 64 keys is walked whole.
#include "common.h"

namespace {
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
constexpr int ROWS = 64;   // query rows per workgroup
constexpr int KEYS = 64;   // keys per tile
constexpr int THREADS = 256;

__device__ __forceinline__ float row4_max(float v) {   // over the 4 lanes l, l ^ 16, l ^ 32, l ^ 48 of a row
  v = fmaxf(v, __shfl_xor(v, 16, WAVE));
  return fmaxf(v, __shfl_xor(v, 32, WAVE));
}
__device__ __forceinline__ float row4_sum(float v) {
  v += __shfl_xor(v, 16, WAVE);
  return v + __shfl_xor(v, 32, WAVE);
}

struct F32Args {
  const int* cu;
  const int* ctx;
  const int* table;
  int n_req, max_pages, page_size, num_pages;
  int page_shift;       // log2(page_size) if it is a power of two, else -1
  int nh, nkv;
  long ldq, ldo;
  float scale;
  int window;
  const float* slopes;  // [nh] or null
  const float* bias;    // [bias_len, nh] or null
  int bias_len;
  const float* sink;    // [nh] or null
  int chunk;
  float softcap;
  int wide_out;         // rows of `out` take 16-byte stores
};

// DT: head size = 16 * DT, of values 16 * VT.  POW2: the page size is a power of two (a shift instead of a division, eight a tile).
template <int DT, bool POW2, int VT>
__global__ __launch_bounds__(THREADS) void attention_f32_kernel(const float* __restrict__ q, const float* __restrict__ kpages,
                                                                const float* __restrict__ vpages, float* __restrict__ out, F32Args a) {
  constexpr int HD = 16 * DT, VD = 16 * VT;
  constexpr int VEC = VT % 4 == 0 ? 4 : VT % 2 == 0 ? 2 : 1;
  typedef __attribute__((__vector_size__(VEC * sizeof(float)))) float floatv;
  constexpr int LD = HD + 4;                                // 16 lanes on 16 rows with 16 bytes each: all 64 banks (head size 64)
  constexpr int LDV = VD + 4;
  constexpr int PER_KEY = HD / 4, PER_VALUE = VD / 4;       // 16-byte chunks of a key and of its value
  constexpr int CHUNKS = KEYS * PER_KEY / THREADS;          // of K per thread and tile: DT
  constexpr int VCHUNKS = KEYS * PER_VALUE / THREADS;       // of V: VT
  static_assert(CHUNKS * THREADS == KEYS * PER_KEY && VCHUNKS * THREADS == KEYS * PER_VALUE, "whole chunks");
  __shared__ __attribute__((aligned(16))) float sK[KEYS][LD];
  __shared__ __attribute__((aligned(16))) float sV[KEYS][LDV];

  const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
  // Which request and which of its tiles: 64 requests at a time, a lane each (one after the other, each a wait for memory, 256 requests of one
  // token and 16 heads of 64 took 160 us behind 10 keys; 69 now)
  int tile = blockIdx.x, r = -1, qlen = 0;
  for (int base = 0; base < a.n_req; base += WAVE) {
    const int i = min(base + lane, a.n_req - 1);
    const int len = base + lane < a.n_req ? a.cu[i + 1] - a.cu[i] : 0;
    int upto = (len + ROWS - 1) / ROWS;      // tiles of these requests up to this one
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
      tile = __builtin_amdgcn_readlane(upto, l) - 1 - tile;  // a request's last rows see the most keys: those workgroups start first
      break;
    }
    tile -= __builtin_amdgcn_readlane(upto, WAVE - 1);
  }
  if (r < 0) return;
  const int lr = lane % 16, g = lane / 16;
  const int head = blockIdx.y, kvh = head / (a.nh / a.nkv);
  const int n0 = a.cu[r] + tile * ROWS, p0 = a.ctx[r] + tile * ROWS;
  const int rows_here = min(ROWS, qlen - tile * ROWS);
  const int* table = a.table + (size_t)r * a.max_pages;

  // the row this lane owns (rows past the last one repeat it, and are not stored)
  const int my_row = min(wave * 16 + lr, rows_here - 1);
  floatx4 qf[DT];
#pragma unroll
  for (int s = 0; s < DT; ++s) qf[s] = *(const floatx4*)(q + (size_t)(n0 + my_row) * a.ldq + (size_t)head * HD + s * 16 + g * 4);
  const int pos_row = p0 + my_row;
  auto first_of = [&](int p) { return a.chunk > 0 ? p - p % a.chunk : (a.window > 0 ? max(0, p - a.window + 1) : 0); };
  const int lo_row = first_of(pos_row);
  const int last_pos = p0 + rows_here - 1;
  const int wave_first = p0 + min(wave * 16, rows_here - 1), wave_last = p0 + min(wave * 16 + 15, rows_here - 1);
  const int wave_lo = first_of(wave_first), wave_lo_last = first_of(wave_last);   // (first_of never falls)

  floatx4 o[VT];
#pragma unroll
  for (int t = 0; t < VT; ++t) o[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  // chunk i of this thread: key (tid + 256 i) / PER_KEY of the tile (of V: / PER_VALUE); keys past the last one repeat it, and are zero in LDS
  int page[CHUNKS], vpage[VT == DT ? 1 : VCHUNKS];
  floatx4 kreg[CHUNKS], vreg[VCHUNKS];
  auto key_of = [&](int kt, int i) { return kt * KEYS + (tid + i * THREADS) / PER_KEY; };
  auto value_of = [&](int kt, int i) { return kt * KEYS + (tid + i * THREADS) / PER_VALUE; };
  auto page_of = [&](int key) { return POW2 ? key >> a.page_shift : key / a.page_size; };
  auto ask_pages = [&](int kt) {
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) page[i] = table[page_of(min(key_of(kt, i), last_pos))];
    if constexpr (VT != DT) {
#pragma unroll
      for (int i = 0; i < VCHUNKS; ++i) vpage[i] = table[page_of(min(value_of(kt, i), last_pos))];
    }
  };
  // the place of key `key` in its page `pg` of the pool (never outside the pool)
  auto slot_of = [&](int pg, int key) {
    return ((size_t)min(max(pg, 0), a.num_pages - 1) * a.nkv + kvh) * a.page_size + (key - page_of(key) * a.page_size);
  };
  auto ask_tile = [&](int kt) {
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
      const size_t off = slot_of(page[i], min(key_of(kt, i), last_pos)) * HD + (tid + i * THREADS) % PER_KEY * 4;
      kreg[i] = *(const floatx4*)(kpages + off);
      if constexpr (VT == DT) vreg[i] = *(const floatx4*)(vpages + off);
    }
    if constexpr (VT != DT) {
#pragma unroll
      for (int i = 0; i < VCHUNKS; ++i)
        vreg[i] = *(const floatx4*)(vpages + slot_of(vpage[i], min(value_of(kt, i), last_pos)) * VD + (tid + i * THREADS) % PER_VALUE * 4);
    }
  };
  auto store_tile = [&](int kt) {
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
      const int c = tid + i * THREADS;
      *(floatx4*)&sK[c / PER_KEY][c % PER_KEY * 4] = key_of(kt, i) <= last_pos ? kreg[i] : zero;
    }
#pragma unroll
    for (int i = 0; i < VCHUNKS; ++i) {
      const int c = tid + i * THREADS;
      *(floatx4*)&sV[c / PER_VALUE][c % PER_VALUE * 4] = value_of(kt, i) <= last_pos ? vreg[i] : zero;
    }
  };

  const int kt_first = first_of(p0) / KEYS, kt_stop = last_pos / KEYS + 1;
  ask_pages(kt_first);
  ask_tile(kt_first);
  ask_pages(min(kt_first + 1, kt_stop - 1));
  for (int kt = kt_first; kt < kt_stop; ++kt) {
    __syncthreads();  // everyone is done with the previous tile
    store_tile(kt);
    __syncthreads();
    ask_tile(min(kt + 1, kt_stop - 1));     // (the last tile is asked for once more: no branch around loads in flight)
    ask_pages(min(kt + 2, kt_stop - 1));
    __builtin_amdgcn_sched_barrier(0);      // the loads stay in flight during the arithmetic
    const int key0 = kt * KEYS;
    if (key0 > wave_last || key0 + KEYS <= wave_lo || wave * 16 >= rows_here) continue;   // (the whole wave)

    // S^T = K Q^T: element i of s4[c] is key c * 16 + g * 4 + i against row lr
    floatx4 s4[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) s4[c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < DT; ++s) {
      floatx4 kf[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) kf[c] = *(const floatx4*)&sK[c * 16 + lr][s * 16 + g * 4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c) s4[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[c][j], qf[s][j], s4[c], 0, 0, 0);
    }
    // (each option its own loop behind one branch: within one loop every element has its own branches)
    auto each = [&](auto f) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) s4[c][i] = f(s4[c][i], key0 + c * 16 + g * 4 + i);
    };
    each([&](float s, int) { return s * a.scale; });
    if (a.softcap > 0.f) each([&](float s, int) { return a.softcap * tanhf(s / a.softcap); });
    if (a.slopes) {
      const float slope = a.slopes[head];
      each([&](float s, int key) { return s + slope * (float)(key - pos_row); });
    }
    if (a.bias) each([&](float s, int key) { return s + a.bias[(size_t)min(max(pos_row - key, 0), a.bias_len - 1) * a.nh + head]; });
    // (tiles that every row of the wave sees whole need no mask; the same for the whole wave, and said so)
    const bool masked = __builtin_amdgcn_readfirstlane((int)(key0 + KEYS - 1 > wave_first || key0 < wave_lo_last)) != 0;
    bool finite = true;
    if (masked) {
      float probe = 0.f;
      each([&](float s, int key) { return key <= pos_row && key >= lo_row ? s : -INFINITY; });
#pragma unroll
      for (int s = 0; s < VT; ++s)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const floatx4 v = *(const floatx4*)&sV[c * 16 + lr][s * 16 + g * 4];
#pragma unroll
          for (int j = 0; j < 4; ++j) probe = fmaf(v[j], 0.f, probe);
        }
      finite = __builtin_amdgcn_ballot_w64(!(probe == 0.f)) == 0;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s4[c][i]);
    const float m_new = fmaxf(m, row4_max(mx));
    const float base = m_new == -INFINITY ? 0.f : m_new;    // no key seen yet: weights of 0, not of NaN
    const float keep = expf(m - base);
    m = m_new;
    l *= keep;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s4[c][i] = expf(s4[c][i] - base);
        l += s4[c][i];
      }
    if (__builtin_amdgcn_ballot_w64(keep != 1.f) != 0) {
#pragma unroll
      for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[t][i] *= keep;
    }
    // O^T += V^T P^T: step (c, i) takes the keys c * 16 + g * 4 + i; tile t = u VEC + e the d = u 16 VEC + VEC (row of the tile) + e
    if (finite) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int u = 0; u < VT / VEC; ++u) {
            const floatv v = *(const floatv*)&sV[c * 16 + g * 4 + i][u * 16 * VEC + lr * VEC];
#pragma unroll
            for (int e = 0; e < VEC; ++e) o[u * VEC + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], s4[c][i], o[u * VEC + e], 0, 0, 0);
          }
    } else {
      // an infinity or a NaN among the values of a tile that some row sees in part: a weight of 0 for a key that a row does
      // not see would make it NaN there, so the keys are taken one by one
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          for (int gg = 0; gg < 4; ++gg) {
            const int row = c * 16 + gg * 4 + i;
            const float w = __shfl(s4[c][i], gg * 16 + lr, WAVE);
            if (key0 + row > pos_row || key0 + row < lo_row) continue;
#pragma unroll
            for (int t = 0; t < VT; ++t)
#pragma unroll
              for (int k = 0; k < 4; ++k) o[t][k] = fmaf(w, sV[row][t / VEC * 16 * VEC + (g * 4 + k) * VEC + t % VEC], o[t][k]);
          }
    }
  }

  l = row4_sum(l);
  if (wave * 16 + lr >= rows_here) return;
  if (a.sink) l += expf(a.sink[head] - m);
  const float inv = 1.0f / l;
  float* dst = out + (size_t)(n0 + my_row) * a.ldo + (size_t)head * VD;
#pragma unroll
  for (int u = 0; u < VT / VEC; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float* to = dst + u * 16 * VEC + (g * 4 + i) * VEC;
      floatv v;
#pragma unroll
      for (int e = 0; e < VEC; ++e) v[e] = o[u * VEC + e][i] * inv;
      if (a.wide_out) {
        *(floatv*)to = v;
      } else {
#pragma unroll
        for (int e = 0; e < VEC; ++e) to[e] = v[e];
      }
    }
}
}  // namespace

GIBBS_EXPORT int gibbs_attention_f32_takes(int hd, int vd) { return hd >= 16 && hd <= 128 && hd % 16 == 0 && (vd == hd || (vd == 2 * hd && hd <= 64)); }

// q: float32 rows (stride ldq), rows of request r are cu[r] .. cu[r + 1] at positions ctx[r] ..; pages [num_pages, nkv, page_size,
// hd] and [num_pages, nkv, page_size, vd] (keys of a multiple of 16 up to 128, values of that size or, for keys up to 64, of twice that); out: row stride ldo.  cu may start above 0 (the requests of a
// step from some request on); n_rows counts the rows from there.  The other operands are gibbs_attention_plain_masked's.
GIBBS_EXPORT int gibbs_attention_f32_values(const void* q, const void* kpages, const void* vpages, void* out, const int* cu, const int* ctx,
                                     const int* table, int n_req, int max_pages, int page_size, int num_pages, int n_rows, int nh,
                                     int nkv, int hd, int vd, long ldq, long ldo, float scale, int window, const float* slopes, const float* bias,
                                     int bias_len, const float* sink, int chunk, float softcap, hipStream_t stream) {
  GIBBS_REQUIRE(n_rows >= 0 && n_req >= 0 && nh > 0 && nkv > 0 && nh % nkv == 0 && nh <= 65535, "attention_f32: bad sizes rows=%d requests=%d heads=%d kv=%d",
                n_rows, n_req, nh, nkv);
  GIBBS_REQUIRE(hd % 16 == 0 && hd >= 16 && hd <= 128, "attention_f32: head size %d must be a multiple of 16 up to 128", hd);
  GIBBS_REQUIRE(gibbs_attention_f32_takes(hd, vd), "attention_f32: values of %d beside keys of %d", vd, hd);
  GIBBS_REQUIRE(ldq % 4 == 0 && ((uintptr_t)q | (uintptr_t)kpages | (uintptr_t)vpages) % 16 == 0, "attention_f32: rows must be 16-byte aligned");
  GIBBS_REQUIRE(ldq >= (long)nh * hd && ldo >= (long)nh * vd, "attention_f32: row strides shorter than heads * hd");
  GIBBS_REQUIRE(page_size > 0 && max_pages > 0 && num_pages > 0 && window >= 0, "attention_f32: bad cache geometry");
  GIBBS_REQUIRE(!bias || bias_len > 0, "attention_f32: an empty table of score biases");
  GIBBS_REQUIRE(chunk >= 0 && !(chunk > 0 && window > 0) && softcap >= 0.f, "attention_f32: a window of %d with chunks of %d, scores capped at %g", window, chunk, softcap);
  if (n_rows == 0 || n_req == 0) return 0;
  const int page_shift = (page_size & (page_size - 1)) == 0 ? __builtin_ctz(page_size) : -1;
  F32Args a{cu, ctx, table, n_req, max_pages, page_size, num_pages, page_shift, nh, nkv, ldq, ldo, scale, window, slopes, bias, bias_len, sink, chunk, softcap,
            ldo % 4 == 0 && (uintptr_t)out % 16 == 0};
  const dim3 grid(ceil_div(n_rows, ROWS) + n_req, nh);
  const float *qq = (const float*)q, *kk = (const float*)kpages, *vv = (const float*)vpages;
  float* oo = (float*)out;
#define F32_ATTENTION(DT, VT)                                                                                         \
  do {                                                                                                                \
    if (page_shift >= 0) attention_f32_kernel<DT, true, VT><<<grid, THREADS, 0, stream>>>(qq, kk, vv, oo, a);          \
    else attention_f32_kernel<DT, false, VT><<<grid, THREADS, 0, stream>>>(qq, kk, vv, oo, a);                         \
  } while (0)
  const bool twice = vd != hd;
  switch (hd / 16) {
    case 1: if (twice) F32_ATTENTION(1, 2); else F32_ATTENTION(1, 1); break;
    case 2: if (twice) F32_ATTENTION(2, 4); else F32_ATTENTION(2, 2); break;
    case 3: if (twice) F32_ATTENTION(3, 6); else F32_ATTENTION(3, 3); break;
    case 4: if (twice) F32_ATTENTION(4, 8); else F32_ATTENTION(4, 4); break;
    case 5: F32_ATTENTION(5, 5); break;
    case 6: F32_ATTENTION(6, 6); break;
    case 7: F32_ATTENTION(7, 7); break;
    default: F32_ATTENTION(8, 8); break;
  }
#undef F32_ATTENTION
  GIBBS_LAUNCH_STATUS("attention_f32");
}

GIBBS_EXPORT int gibbs_attention_f32(const void* q, const void* kpages, const void* vpages, void* out, const int* cu, const int* ctx,
                                     const int* table, int n_req, int max_pages, int page_size, int num_pages, int n_rows, int nh,
                                     int nkv, int hd, long ldq, long ldo, float scale, int window, const float* slopes, const float* bias,
                                     int bias_len, const float* sink, int chunk, float softcap, hipStream_t stream) {
  return gibbs_attention_f32_values(q, kpages, vpages, out, cu, ctx, table, n_req, max_pages, page_size, num_pages, n_rows, nh, nkv, hd, hd, ldq, ldo, scale,
                                    window, slopes, bias, bias_len, sink, chunk, softcap, stream);
}
