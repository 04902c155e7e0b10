// wave_ops.hpp -- sums over the lanes of a wave with DPP moves.  gfx950, wave64.
//
// __shfl_xor goes through the LDS crossbar (ds_bpermute, about 64 clocks a
// 32-bit word); a DPP move is a VALU operand modifier (a few clocks).  A wave sum
// of one double takes about 0.35 us as a butterfly of shuffles and 0.08 us here,
// which matters where a solve waits on it twice an iteration.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace onsas {

// quad_perm [1,0,3,2] and [2,3,0,1], row_half_mirror, row_mirror: each pairs a
// lane with one outside the group (of 1, 2, 4, 8 lanes) summed so far
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140;
constexpr int kDppRor8 = 0x128;  // row_ror:8, lane ^ 8 of a row of 16

template <int CTRL>
__device__ inline float dpp_move(float x) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ inline double dpp_move(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

// the value of lane C of the caller's group of four
template <int C, typename T>
__device__ inline T quad_lane(T x) {
  return dpp_move<C | (C << 2) | (C << 4) | (C << 6)>(x);
}

// sum over groups of W = 2, 4, 8 or 16 consecutive lanes, in every lane of them
template <int W, typename T>
__device__ inline T group_sum(T x) {
  if (W >= 2) x += dpp_move<kDppXor1>(x);
  if (W >= 4) x += dpp_move<kDppXor2>(x);
  if (W >= 8) x += dpp_move<kDppHalfMirror>(x);
  if (W >= 16) x += dpp_move<kDppMirror>(x);
  return x;
}

__device__ inline float read_lane(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}
__device__ inline double read_lane(double x, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), l),
                          __builtin_amdgcn_readlane(__double2loint(x), l));
}

// sum over the wave, in every lane (all 64 lanes active)
__device__ inline double wave_sum(double x) {
  x = group_sum<16>(x);
  return (read_lane(x, 0) + read_lane(x, 16)) + (read_lane(x, 32) + read_lane(x, 48));
}

}  // namespace onsas
