// Shared declarations of the gfx950 kernels: element types, the error channel that the
// Python side reads, and small wave/block reductions (64-wide wavefronts).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>
#include <type_traits>

typedef __bf16 bf16;

// Element type tags passed across the C interface.
enum { GIBBS_F32 = 0, GIBBS_BF16 = 1 };

#define GIBBS_EXPORT extern "C" __attribute__((visibility("default")))

// Records a message for gibbs_last_error() and returns a non-zero status.
int gibbs_fail(const char* fmt, ...);

#define GIBBS_REQUIRE(cond, ...)                 \
  do {                                           \
    if (!(cond)) return gibbs_fail(__VA_ARGS__); \
  } while (0)

// Status of the launch that was just queued.
#define GIBBS_LAUNCH_STATUS(what)                                                      \
  do {                                                                                 \
    hipError_t e_ = hipGetLastError();                                                 \
    if (e_ != hipSuccess) return gibbs_fail("%s: %s", what, hipGetErrorString(e_));    \
    return 0;                                                                          \
  } while (0)

static inline int ceil_div(long a, long b) { return (int)((a + b - 1) / b); }

__device__ __forceinline__ float to_float(float v) { return v; }
__device__ __forceinline__ float to_float(bf16 v) { return (float)v; }
template <typename T> __device__ __forceinline__ T from_float(float v);
template <> __device__ __forceinline__ float from_float<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16 from_float<bf16>(float v) { return (bf16)v; }

constexpr int WAVE = 64;

// What lane (lane ^ MASK) holds, by moves between lanes of the vector units (4 to 12 cycles) instead of a trip through LDS (some 120,
// and such exchanges come six in a row).  All 64 lanes take part.
template <int MASK>
__device__ __forceinline__ uint32_t lane_xor_bits(uint32_t v) {
  static_assert(MASK == 1 || MASK == 2 || MASK == 4 || MASK == 8 || MASK == 16 || MASK == 32, "one bit of the lane's number");
  if constexpr (MASK >= 16) {
    const auto both = [&] {
      if constexpr (MASK == 32) return __builtin_amdgcn_permlane32_swap(v, v, false, false);
      else return __builtin_amdgcn_permlane16_swap(v, v, false, false);
    }();      // [0]: of each pair of halves the lower one's value in both, [1]: the upper one's
    return (threadIdx.x & MASK) ? both[0] : both[1];
  } else if constexpr (MASK == 4) {      // (lane i -> 7 - i, then quads reversed: i -> i ^ 7 ^ 3)
    return __builtin_amdgcn_update_dpp(0, __builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true), 0x1B, 0xf, 0xf, true);
  } else {
    constexpr int CTRL = MASK == 1 ? 0xB1 : (MASK == 2 ? 0x4E : 0x128);      // quad_perm [1,0,3,2], [2,3,0,1], row_ror:8
    return __builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
  }
}
template <int MASK>
__device__ __forceinline__ float lane_xor_float(float v) { return __uint_as_float(lane_xor_bits<MASK>(__float_as_uint(v))); }
// f(v, what lane ^ 32 has), then lane ^ 16, 8, 4, 2, 1: every lane gets the same result of a commutative f.
template <typename T, typename F>
__device__ __forceinline__ T wave_fold(T v, F f) {
  static_assert(sizeof(T) == 4, "a register");
  const auto bits = [](T x) { return __builtin_bit_cast(uint32_t, x); };
  const auto from = [](uint32_t x) { return __builtin_bit_cast(T, x); };
  const auto a = __builtin_amdgcn_permlane32_swap(bits(v), bits(v), false, false);
  v = f(from(a[0]), from(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(bits(v), bits(v), false, false);
  v = f(from(b[0]), from(b[1]));
  v = f(v, from(lane_xor_bits<8>(bits(v))));
  v = f(v, from(lane_xor_bits<4>(bits(v))));
  v = f(v, from(lane_xor_bits<2>(bits(v))));
  return f(v, from(lane_xor_bits<1>(bits(v))));
}
__device__ __forceinline__ float wave_sum(float v) {
  return wave_fold(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_max(float v) {
  return wave_fold(v, [](float a, float b) { return fmaxf(a, b); });
}

// 16 bytes a lane from memory to LDS without registers: from base + at (the same in all lanes) + lane_at, to lds + 16 x lane.  `bytes` from base are there;
// beyond, zeros come.  A buffer load, not a global one: beside a global load to LDS the compiler waits for all LDS reads wherever it waits for one.
__device__ __forceinline__ void buffer_to_lds(const void* base, uint32_t bytes, uint32_t at, uint32_t lane_at, void* lds) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the host's pass does not know the builtin)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00020000),
                                           (__attribute__((address_space(3))) void*)lds, 16, (int)lane_at, (int)at, 0, 0);
#endif
}
// A barrier behind which the wave's LDS reads and all but the last LEFT of its loads are through.  Known to the compiler (waits in assembler are not, and it
// waits once more), and without the wait for every load that __syncthreads() is.
template <int LEFT>
__device__ __forceinline__ void barrier_behind_loads() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((LEFT & 15) | LEFT >> 4 << 14 | 7 << 4);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Sum over a block of up to 1024 threads; every thread gets the result.  `scratch` holds
// one float per wave.  The order of additions is fixed by the thread layout alone.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  v = wave_sum(v);
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int n_waves = (blockDim.x + WAVE - 1) / WAVE;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  // (read side by side where their number is a usual one: one by one they were a tenth of a microsecond each)
  auto together = [&](auto count) {
    float part[decltype(count)::value], total = 0.f;
#pragma unroll
    for (int i = 0; i < decltype(count)::value; ++i) part[i] = scratch[i];
#pragma unroll
    for (int i = 0; i < decltype(count)::value; ++i) total += part[i];
    return total;
  };
  if (n_waves == 8) return together(std::integral_constant<int, 8>{});
  if (n_waves == 4) return together(std::integral_constant<int, 4>{});
  float total = 0.f;
  for (int i = 0; i < n_waves; ++i) total += scratch[i];
  return total;
}

// first + part[apart] + part[2 apart] + ... (`more` of them), in this order, read from LDS eight or four at a time: one by one each is a
// trip of its own, 60 ns.
__device__ __forceinline__ float strided_sum(float first, const float* part, int more, int apart) {
  auto some = [&](auto count, int g) {
    constexpr int N = decltype(count)::value;
    float m[N];
#pragma unroll
    for (int u = 0; u < N; ++u) m[u] = part[min(g + u, more) * apart];
#pragma unroll
    for (int u = 0; u < N; ++u) first = g + u <= more ? first + m[u] : first;
  };
  int g = 1;
  for (; more - g >= 4; g += 8) some(std::integral_constant<int, 8>{}, g);
  if (g <= more) some(std::integral_constant<int, 4>{}, g);
  return first;
}

// Every file of the library sees the entry points' prototypes, so that a definition whose signature has
// drifted from what the native step (step_plan.hip) calls does not compile.
#include "kernels.h"
