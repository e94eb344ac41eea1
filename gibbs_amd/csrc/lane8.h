// Helpers for kernels in which a lane holds 8 consecutive bfloat16 elements (16 bytes) of a head
// and LPK neighbouring lanes hold the head: sums over the lane group, per-head RMSNorm and rotary
// position encoding in that layout.
#pragma once
#include "common.h"
#include <type_traits>

constexpr int EPL = 8;  // head-dim elements per lane (16 bytes of bfloat16)

// Cosine and sine of a rotation angle: the one place that computes them, so that the table and
// every kernel that rotates beyond the table agree to the bit.
__device__ __forceinline__ void rope_cos_sin(float angle, float* c, float* s) {
  *c = cosf(angle);
  *s = sinf(angle);
}

__device__ __forceinline__ void unpack8(const uint4& raw, float* f) {
  const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(w[i] << 16);
    f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
}

__device__ __forceinline__ uint4 pack8(const float* f) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bf16 lo = (bf16)f[2 * i], hi = (bf16)f[2 * i + 1];
    w[i] = (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// Sum over the LPK neighbouring lanes that share a key, every one of them getting the total.
// Data-parallel-primitive moves (a few cycles each) instead of LDS permutes (tens of cycles each,
// and this sum sits on the critical path of every key): swap within pairs, within quads, then
// mirror the half row (lane i <-> 7 - i: the other quad) and the row (i <-> 15 - i: the other half).
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int LPK>
__device__ __forceinline__ float group_sum(float v) {
  if (LPK >= 2) v += dpp_move<0xB1>(v);   // quad_perm [1,0,3,2]
  if (LPK >= 4) v += dpp_move<0x4E>(v);   // quad_perm [2,3,0,1]
  if (LPK >= 8) v += dpp_move<0x141>(v);  // row_half_mirror
  if (LPK >= 16) v += dpp_move<0x140>(v); // row_mirror
  if (LPK >= 32) v += __shfl_xor(v, 16, WAVE);
  return v;
}

// The value of lane (lane ^ MASK), MASK 1, 2, 4 or 8, likewise without LDS.
template <int MASK>
__device__ __forceinline__ float lane_xor(float v) {
  static_assert(MASK == 1 || MASK == 2 || MASK == 4 || MASK == 8, "inside a row of 16 lanes");
  if (MASK == 1) return dpp_move<0xB1>(v);
  if (MASK == 2) return dpp_move<0x4E>(v);
  if (MASK == 4) return dpp_move<0x1B>(dpp_move<0x141>(v));   // (i -> 7 - i, then quad_perm [3,2,1,0]: i -> i ^ 7 ^ 3)
  return dpp_move<0x128>(v);                                  // (row_ror:8)
}
// The sum of a head's squares with its 8 LPK elements 8 to a lane, to the bit as a wave with one element a lane makes it (lane l: the squares of
// elements l and l + 64 in that order, then wave_sum): kernels of both layouts give a head the same norm.  Element 8 j + i is lane j's value
// i, so wave_sum's halves, quarters and eighths are lanes, and what it adds last are the values inside a lane.  Every such step over lanes
// halves the values that a lane still has instead of adding all of them twice (a + b and b + a are the same bits), so that 10 moves do for 8
// values in 8 lanes where a sum of each lane's own total takes 3.
template <int LPK>
__device__ __forceinline__ float head_squares(const float* v, int lane) {
  static_assert(LPK == 2 || LPK == 4 || LPK == 8 || LPK == 16, "heads of 16, 32, 64 or 128");
  float s[8];
  if constexpr (LPK == 16) {        // elements l and l + 64 lie 8 lanes apart: each of the two lanes takes four of the eight pairs
    const bool low = (lane & 8) == 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float own = low ? v[i] : v[4 + i], got = lane_xor<8>(low ? v[4 + i] : v[i]);
      const float first = low ? own : got, second = low ? got : own;
      s[i] = fmaf(second, second, fmaf(first, first, 0.f));
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] = fmaf(v[i], v[i], 0.f);
  }
  // a lane with the bit set goes on with the upper half of its N values
  auto halve = [&](auto mask, auto count) {
    constexpr int M = decltype(mask)::value, H = decltype(count)::value / 2;
    const bool low = (lane & M) == 0;
#pragma unroll
    for (int i = 0; i < H; ++i) {
      const float give = low ? s[H + i] : s[i], own = low ? s[i] : s[H + i];
      s[i] = own + lane_xor<M>(give);
    }
  };
  auto add = [&](auto mask, auto count) {
#pragma unroll
    for (int i = 0; i < decltype(count)::value; ++i) s[i] += lane_xor<decltype(mask)::value>(s[i]);
  };
  using std::integral_constant;
  integral_constant<int, 1> one;
  integral_constant<int, 2> two;
  integral_constant<int, 4> four;
  integral_constant<int, 8> eight;
  if constexpr (LPK == 16) {
    halve(four, four);
    halve(two, two);
    add(one, one);
    add(eight, one);      // (the values of a lane: those of 4, 2 and 1 apart, which the halvings put into lanes)
    add(four, one);
    add(two, one);
    return s[0];
  } else if constexpr (LPK == 8) {
    halve(four, eight);
    halve(two, four);
    halve(one, two);
    add(four, one);
    add(two, one);
    add(one, one);
    return s[0];
  } else if constexpr (LPK == 4) {
    halve(two, eight);
    halve(one, four);
    add(two, two);
    add(one, two);
    return s[0] + s[1];
  } else {
    halve(one, eight);
    add(one, four);
    return (s[0] + s[2]) + (s[1] + s[3]);
  }
}

__device__ __forceinline__ bool finite(float x) { return x * 0.f == 0.f; }
// For an operand of a product whose other operand has zeros above a diagonal (lane (g, c) of a wave: rows 4 g .. 4 g + 3 of column c of a 16 x
// 16 tile): what is not finite is taken out of it, since 0 times that would reach the rows in front of it too.  Returned is what
// to add to the product: NaN in the rows from the first such one of its column on, else 0.
template <typename F4>
__device__ __forceinline__ F4 nan_behind(F4& x, int g) {
  F4 add = {0.f, 0.f, 0.f, 0.f};
  if (__builtin_amdgcn_ballot_w64(!finite(x[0] * 0.f + x[1] * 0.f + x[2] * 0.f + x[3] * 0.f)) != 0) {
    float run = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      run += x[i] * 0.f;
      add[i] = run;
      if (!finite(x[i])) x[i] = 0.f;
    }
    float before = 0.f;
#pragma unroll
    for (int o = 1; o < 4; ++o) {
      const float y = __shfl_up(run, 16 * o, WAVE);
      if (g >= o) before += y;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) add[i] += before;
  }
  return add;
}

// Rotation factors of this lane's 8 elements at position `pos` (the same for every head).
struct Rot8 {
  float c[EPL], s[EPL];
};

// `table`: (cos, sin) of positions 0 .. table_len-1, [table_len, rot/2], made by rope_table from the
// same float32 angles with the same functions; later positions are computed here.
__device__ __forceinline__ Rot8 rotation8(int e0, const float* inv_freq, int rot, int variant, int pos,
                                          const float2* table, int table_len) {
  Rot8 r;
  const int half = rot / 2;
  const bool tabled = table && pos < table_len;
  // (eight elements of the rotated part have neighbouring factors: a table's row is read 16 bytes at a time, not a pair at a time under
  // a condition of its own.  The table is of pairs, its rows need not start at 16 bytes)
  typedef float floatx4_8 __attribute__((ext_vector_type(4), aligned(8)));
  if (inv_freq && tabled && e0 + EPL <= rot && half % EPL == 0) {
    const float2* row = table + (size_t)pos * half + (variant == 1 ? e0 / 2 : (e0 < half ? e0 : e0 - half));
    if (variant == 1) {
#pragma unroll
      for (int i = 0; i < EPL; i += 4) {
        const floatx4_8 t = *(const floatx4_8*)(row + i / 2);
        r.c[i] = r.c[i + 1] = t[0]; r.s[i] = r.s[i + 1] = t[1];
        r.c[i + 2] = r.c[i + 3] = t[2]; r.s[i + 2] = r.s[i + 3] = t[3];
      }
    } else {
#pragma unroll
      for (int i = 0; i < EPL; i += 2) {
        const floatx4_8 t = *(const floatx4_8*)(row + i);
        r.c[i] = t[0]; r.s[i] = t[1]; r.c[i + 1] = t[2]; r.s[i + 1] = t[3];
      }
    }
    return r;
  }
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    const int e = e0 + i;
    r.c[i] = 1.f;
    r.s[i] = 0.f;
    if (inv_freq && e < rot) {
      const int j = variant == 1 ? e / 2 : (e < half ? e : e - half);
      if (tabled) {
        const float2 cs = table[(size_t)pos * half + j];
        r.c[i] = cs.x;
        r.s[i] = cs.y;
      } else {
        rope_cos_sin((float)pos * inv_freq[j], &r.c[i], &r.s[i]);
      }
    }
  }
  return r;
}

// Norm (optional) and rotation of one head held 8 elements per lane by LPK neighbouring lanes.
// `v` are this lane's elements e0 .. e0+7 of the head; returns them normed and rotated.
// `gain8`: the norm's gain for this lane's elements, already in registers (a caller that norms several heads
// reads it once); `normed` false: no norm.
template <int LPK>
__device__ __forceinline__ void norm_rope8_with(float* v, int e0, int hd, bool normed, const float* gain8, float eps,
                                                bool rotate, const Rot8& rt, int rot, int variant, int lane) {
  const bool active = e0 < hd;
  if (normed) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < EPL; ++i) ss += v[i] * v[i];
    ss = group_sum<LPK>(ss);
    const float sc = 1.0f / sqrtf(ss / (float)hd + eps);
#pragma unroll
    for (int i = 0; i < EPL; ++i) v[i] = active ? v[i] * sc * gain8[i] : 0.f;
  }
  if (!rotate) return;
  const int half = rot / 2;
  if (variant == 1) {  // pairs (2j, 2j+1) lie in one lane
#pragma unroll
    for (int i = 0; i < EPL; i += 2) {
      if (e0 + i + 1 < rot) {
        const float x0 = v[i], x1 = v[i + 1];
        v[i] = x0 * rt.c[i] - x1 * rt.s[i];
        v[i + 1] = x0 * rt.s[i] + x1 * rt.c[i];
      }
    }
    return;
  }
  // half split: element e pairs with e + half (e < half) or e - half; the partner lies half/8 lanes away
  const int shift = half / EPL;  // half is a multiple of 8 (rotary sizes in steps of 16)
  const int base = lane - lane % LPK;
  const int sub = lane % LPK;
  const bool low = e0 < half;
  const int partner = base + (low ? sub + shift : sub - shift);
  const int src = (partner >= base && partner < base + LPK) ? partner : lane;
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    const float other = __shfl(v[i], src, WAVE);
    if (e0 + i < rot) v[i] = low ? v[i] * rt.c[i] - other * rt.s[i] : other * rt.s[i] + v[i] * rt.c[i];
  }
}

// The same with the gain read here (null: no norm).
template <int LPK>
__device__ __forceinline__ void norm_rope8(float* v, int e0, int hd, const float* gain, float eps, bool rotate,
                                           const Rot8& rt, int rot, int variant, int lane) {
  float gain8[EPL];
#pragma unroll
  for (int i = 0; i < EPL; ++i) gain8[i] = (gain && e0 < hd) ? gain[e0 + i] : 1.f;
  norm_rope8_with<LPK>(v, e0, hd, gain != nullptr, gain8, eps, rotate, rt, rot, variant, lane);
}
