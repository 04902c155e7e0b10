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

// Values that are to be loaded before a branch that does not need them.  A load
// whose result is used only behind an early return is moved there by the compiler,
// so the flag's round trip comes first and the load's after it; here the values
// (wave-uniform ones in s, others in v) and the flag arrive together.
__device__ inline void arrive_s(int32_t& a, int32_t& b, int32_t& flag) {
  a = __builtin_amdgcn_readfirstlane(a);
  b = __builtin_amdgcn_readfirstlane(b);
  flag = __builtin_amdgcn_readfirstlane(flag);
  asm volatile("" : "+s"(a), "+s"(b), "+s"(flag));
}
__device__ inline void arrive_v(int32_t& a, int32_t& b, int32_t& flag) {
  flag = __builtin_amdgcn_readfirstlane(flag);
  asm volatile("" : "+v"(a), "+v"(b), "+s"(flag));
}

// The index of a clamped slot: loaded whether or not the slot counts (else the
// compiler puts its load, and the gather behind it, under the slot's condition,
// one round trip after the other).
template <int N>
__device__ inline void arrive_all(int32_t (&x)[N]) {
#pragma unroll
  for (int q = 0; q < N; ++q) asm volatile("" : "+v"(x[q]));
}

// quad_perm [1,0,3,2] and [2,3,0,1], row_half_mirror, row_mirror: each pairs a
// lane with one outside the group (of 1, 2, 4, 8 lanes) summed so far
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140;
constexpr int kDppRor = 0x120;  // + n: row_ror:n, rotations within a row of 16 lanes

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

// x + x of lane ^ 16 and lane ^ 32 (VALU row swaps)
__device__ inline float xor16_sum(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ inline float xor32_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ inline double xor16_sum(double x) {
  const uint32_t l = (uint32_t)__double2loint(x), h = (uint32_t)__double2hiint(x);
  const auto a = __builtin_amdgcn_permlane16_swap(l, l, false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(h, h, false, false);
  return __hiloint2double((int)b[0], (int)a[0]) + __hiloint2double((int)b[1], (int)a[1]);
}
__device__ inline double xor32_sum(double x) {
  const uint32_t l = (uint32_t)__double2loint(x), h = (uint32_t)__double2hiint(x);
  const auto a = __builtin_amdgcn_permlane32_swap(l, l, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(h, h, false, false);
  return __hiloint2double((int)b[0], (int)a[0]) + __hiloint2double((int)b[1], (int)a[1]);
}

// sum over groups of 32 or 64 consecutive lanes, in every lane of them
template <int W, typename T>
__device__ inline T half_or_wave_sum(T x) {
  x = xor16_sum(group_sum<16>(x));
  return W == 64 ? xor32_sum(x) : x;
}
// sum over the lanes of equal index modulo S = 2, 4 or 8
template <int S, typename T>
__device__ inline T stride_sum(T x) {
  x += dpp_move<kDppRor + 8>(x);
  if (S <= 4) x += dpp_move<kDppRor + 4>(x);
  if (S <= 2) x += dpp_move<kDppRor + 2>(x);
  return xor32_sum(xor16_sum(x));
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
