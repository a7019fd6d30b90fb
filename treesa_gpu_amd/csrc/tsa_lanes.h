// tsa_lanes.h -- exchanges between lanes of a wave without LDS.
//
// __shfl_xor is a ds_bpermute: an LDS round trip (about 130 cycles) and an address computation a step.  On gfx950 the
// same exchanges are vector instructions: DPP permutes inside a row of 16 lanes, v_permlane16_swap / v_permlane32_swap
// across rows and halves.
#pragma once
#include <stdint.h>
#include <hip/hip_runtime.h>

// x of lane ^ O.  Both lanes of a pair must be active.
template <int O>
__device__ __forceinline__ uint32_t tsa_lane_xor(uint32_t x) {
  static_assert(O == 1 || O == 2 || O == 4 || O == 8 || O == 16 || O == 32, "a power of two below 64");
  const int v = (int)x;
  if constexpr (O == 1) return (uint32_t)__builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true);   // quad_perm [1, 0, 3, 2]
  if constexpr (O == 2) return (uint32_t)__builtin_amdgcn_mov_dpp(v, 0x4E, 0xf, 0xf, true);   // quad_perm [2, 3, 0, 1]
  if constexpr (O == 4)  // half-row mirror (lane ^ 7), then each quad reversed (lane ^ 3)
    return (uint32_t)__builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(v, 0x141, 0xf, 0xf, true), 0x1B, 0xf, 0xf, true);
  if constexpr (O == 8) return (uint32_t)__builtin_amdgcn_mov_dpp(v, 0x128, 0xf, 0xf, true);  // row rotated by 8
  if constexpr (O == 16) {
    // the first operand's odd rows against the second's even ones: {rows 0 0 2 2, rows 1 1 3 3}
    const auto p = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return (__lane_id() & 16u) ? p[0] : p[1];
  }
  if constexpr (O == 32) {
    const auto p = __builtin_amdgcn_permlane32_swap(x, x, false, false);  // {low half twice, high half twice}
    return (__lane_id() & 32u) ? p[0] : p[1];
  }
  return x;
}
template <int O>
__device__ __forceinline__ int tsa_lane_xor(int x) { return (int)tsa_lane_xor<O>((uint32_t)x); }
template <int O>
__device__ __forceinline__ float tsa_lane_xor(float x) { return __uint_as_float(tsa_lane_xor<O>(__float_as_uint(x))); }
template <int O>
__device__ __forceinline__ uint64_t tsa_lane_xor(uint64_t x) {
  return ((uint64_t)tsa_lane_xor<O>((uint32_t)(x >> 32)) << 32) | tsa_lane_xor<O>((uint32_t)x);
}

// f(std::integral_constant<int, O>) for O = N/2, N/4, ..., 1: a butterfly over N lanes.
template <int O>
struct TsaLaneStep {
  static constexpr int value = O;
};
template <int N, class F>
__device__ __forceinline__ void tsa_lane_butterfly(F f) {
  if constexpr (N > 1) {
    f(TsaLaneStep<N / 2>{});
    tsa_lane_butterfly<N / 2>(f);
  }
}
// Sum and maximum over N lanes, in every lane.
template <int N>
__device__ __forceinline__ int tsa_lane_sum(int x) {
  tsa_lane_butterfly<N>([&](auto o) { x += tsa_lane_xor<decltype(o)::value>(x); });
  return x;
}
template <int N>
__device__ __forceinline__ int tsa_lane_max(int x) {
  tsa_lane_butterfly<N>([&](auto o) {
    const int y = tsa_lane_xor<decltype(o)::value>(x);
    x = x > y ? x : y;
  });
  return x;
}
