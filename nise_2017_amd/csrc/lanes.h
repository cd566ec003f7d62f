// Sums across the lanes of a wave by DPP and the row-swap instructions
// (VALU only; __shfl_xor goes through the LDS crossbar, a round trip of
// about 100 cycles per level).
#pragma once

#include <hip/hip_runtime.h>

namespace nise {

template <int kCtrl>
__device__ __forceinline__ float dpp_move(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, 0xF, 0xF, false));
}
// x of the row 16 lanes away (lane ^ 16) plus the lane's own, and lane ^ 32.
__device__ __forceinline__ float add_xor16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float add_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// Sum over the aligned groups of W lanes (W a power of two), in every lane.
// Within a row of 16: quad_perm for lane ^ 1 and ^ 2, then the mirrors of 8
// and 16 lanes, whose partners hold the other half's sum.
template <int W>
__device__ __forceinline__ float group_sum(float x) {
  if constexpr (W > 1) x += dpp_move<0xB1>(x);
  if constexpr (W > 2) x += dpp_move<0x4E>(x);
  if constexpr (W > 4) x += dpp_move<0x141>(x);
  if constexpr (W > 8) x += dpp_move<0x140>(x);
  if constexpr (W > 16) x = add_xor16(x);
  if constexpr (W > 32) x = add_xor32(x);
  return x;
}
// Sum over the lanes with the same lane % W (W a power of two), in every
// lane: rotations of 8 and 4 lanes within a row keep lane % 4, then quads.
template <int W>
__device__ __forceinline__ float stride_sum(float x) {
  if constexpr (W <= 8) x += dpp_move<0x128>(x);  // row_ror:8
  if constexpr (W <= 4) x += dpp_move<0x124>(x);  // row_ror:4
  if constexpr (W <= 2) x += dpp_move<0x4E>(x);   // lane ^ 2
  if constexpr (W <= 1) x += dpp_move<0xB1>(x);   // lane ^ 1
  if constexpr (W <= 16) x = add_xor16(x);
  if constexpr (W <= 32) x = add_xor32(x);
  return x;
}

}  // namespace nise
