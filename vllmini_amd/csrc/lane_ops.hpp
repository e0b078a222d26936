// lane_ops.hpp — values of other lanes of a wave without the trip through the LDS unit that a shuffle (ds_bpermute) is: rows of 16 lanes and halves of 32 change
// places by v_permlane16/32_swap, inside a row of 16 the DPP rotations and quad permutes are operands of the arithmetic itself.
//
// A reduction over 64 lanes is six dependent steps; as shuffles each waits for the LDS unit, and a decode step's kernels, chains of latencies of 3 - 7 us, hold two
// to four such reductions.  The partners of every step are those of the shuffles (lane ^ 32, 16, 8, 4, 2, 1 in that order), so sums
// keep every bit: after the step over 8 a row's value repeats every 8 lanes, so a rotation by 4 is the exchange over 4, and so on.
// The lanes that a value is over have to be active: the row's 16 for LANES = 16, the quad's for sum_quad, the wave's for the others, whose rows and halves change places.  Shuffles -> here: paged attention of 32 sequences of 1 - 132 tokens, 12 heads of 64 6.37 -> 5.85 us, of one of 70 3.75 -> 3.50
// (an empty launch: 1.7); decode of GPT-2 small, 32 sequences, 1.5 per cent of a step; width 1024 behind norms, 12 rows, 2 per cent.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vmi_lanes {

template <int CTRL, typename T>
__device__ __forceinline__ T dpp(T v) {
  return __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// op(v, v of lane ^ 16), op(v, v of lane ^ 32); op commutes
template <typename T, typename F>
__device__ __forceinline__ T across16(T v, F op) {
  const uint32_t a = __builtin_bit_cast(uint32_t, v);
  const auto s = __builtin_amdgcn_permlane16_swap(a, a, false, false);
  return op(__builtin_bit_cast(T, (uint32_t)s[0]), __builtin_bit_cast(T, (uint32_t)s[1]));
}
template <typename T, typename F>
__device__ __forceinline__ T across32(T v, F op) {
  const uint32_t a = __builtin_bit_cast(uint32_t, v);
  const auto s = __builtin_amdgcn_permlane32_swap(a, a, false, false);
  return op(__builtin_bit_cast(T, (uint32_t)s[0]), __builtin_bit_cast(T, (uint32_t)s[1]));
}

// over LANES consecutive lanes (16, 32 or the wave's 64), the result in each of them
template <int LANES, typename T, typename F>
__device__ __forceinline__ T over_lanes(T v, F op) {
  static_assert(LANES == 16 || LANES == 32 || LANES == 64, "a row, a half or a wave");
  if constexpr (LANES == 64) v = across32(v, op);
  if constexpr (LANES >= 32) v = across16(v, op);
  v = op(v, dpp<0x128>(v));   // row_ror:8
  v = op(v, dpp<0x124>(v));   // row_ror:4
  v = op(v, dpp<0x122>(v));   // row_ror:2
  return op(v, dpp<0x121>(v));   // row_ror:1
}
template <int LANES>
__device__ __forceinline__ float sum_over(float v) {
  return over_lanes<LANES>(v, [](float a, float b) { return a + b; });
}
template <int LANES>
__device__ __forceinline__ float max_over(float v) {
  return over_lanes<LANES>(v, [](float a, float b) { return fmaxf(a, b); });
}

// sum over the lanes that agree in lane % N, N = 8, 16 or 32
template <int N>
__device__ __forceinline__ float sum_above(float v) {
  auto add = [](float a, float b) { return a + b; };
  if constexpr (N <= 8) v = add(v, dpp<0x128>(v));
  if constexpr (N <= 16) v = across16(v, add);
  return across32(v, add);
}
// sum over N consecutive lanes, N = 1, 2 or 4
template <int N>
__device__ __forceinline__ float sum_quad(float v) {
  static_assert(N == 1 || N == 2 || N == 4, "inside a quad");
  if constexpr (N >= 2) v += dpp<0xB1>(v);   // quad_perm [1,0,3,2]
  if constexpr (N >= 4) v += dpp<0x4E>(v);   // quad_perm [2,3,0,1]
  return v;
}

}  // namespace vmi_lanes
