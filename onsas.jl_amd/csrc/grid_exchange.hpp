// grid_exchange.hpp -- sums and vectors shared by the workgroups of one resident
// launch (the solver kernels that run a whole solve in one launch).  gfx950.
//
// Every workgroup of such a launch is resident at once (the host keeps the grid
// far below the 256 CUs), so workgroups may wait for one another.  A grid-wide
// sum is one exchange: each workgroup writes its partial into its own slot and
// polls the slots of all others.  The slot words are 8 bytes, (epoch << 32) |
// half of the double, so a word carries its own "ready" mark and the sum is
// exact; the partials are added by a fixed tree, the same in every workgroup,
// so all of them take the same branches and a solve is bit-identical from run
// to run.  Measured on one MI355X: 1.2 us for 1 to 8 workgroups, 2.0 us for 32,
// 3.3 us for 128, against 4 to 8 us for a kernel boundary with its drain,
// launch and first loads.
//
// Everything shared goes through relaxed device-scope atomics (they bypass the
// per-XCD L2s), and a workgroup's vector stores are complete (vmcnt 0, then the
// barrier, DRAIN below) before its partial is published, so no L2
// write-back or invalidation is needed and the read-only data stays cached.
// Waits are bounded: a workgroup that polls past `limit` clock ticks (or sees
// another's abort) raises the abort word and the launch drains; the host then
// solves with the one-kernel-per-step path.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "wave_ops.hpp"

namespace onsas {

constexpr int kMaxGridWg = 128;  // workgroups of a resident launch (two polled slots per lane)
constexpr size_t kGridSlotWords = 6 * kMaxGridWg;  // the PCG's slots: a one- and a two-value sum

template <typename T>
__device__ inline T agent_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ inline void agent_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// this wave's stores have reached the device-coherent level
__device__ inline void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

struct GridSlots {
  unsigned long long* words;  // kMaxGridWg slots of the sum's 2 NV words each
  int nwg;
  int* abort;                 // device word: nonzero once a wait has expired
  long long limit;            // ticks of the 100 MHz clock a wait may take
};

// Sum over the workgroup: over each wave, then over the wave partials in index
// order (T threads; sh: NV * T / 64 doubles).  With DRAIN the workgroup's
// earlier stores are complete when the barrier inside opens.  A caller that
// reuses sh has a barrier between two uses.
template <int NV, int T, bool DRAIN>
__device__ inline void wg_partials(double (&v)[NV], double* sh) {
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] = wave_sum(v[q]);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int q = 0; q < NV; ++q) sh[q * (T / 64) + (threadIdx.x >> 6)] = v[q];
  if (DRAIN) stores_done();
  __syncthreads();
}
template <int NV, int T>
__device__ inline void wg_total(double (&v)[NV], const double* sh) {
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    double s = sh[q * (T / 64)];
#pragma unroll
    for (int w = 1; w < T / 64; ++w) s += sh[q * (T / 64) + w];
    v[q] = s;
  }
}
template <int NV, int T>
__device__ inline void wg_sum(double (&v)[NV], double* sh) {
  wg_partials<NV, T, false>(v, sh);
  wg_total<NV, T>(v, sh);
}

// One value of a slot: its two words once both carry the epoch; false once the
// launch is aborted.
template <int NW>
__device__ inline bool poll_words(const unsigned long long* s, uint32_t epoch, const GridSlots& gs,
                                  unsigned long long (&w)[NW]) {
  long long t0 = 0;
  for (uint32_t spin = 0;; ++spin) {
    bool ready = true;
#pragma unroll
    for (int q = 0; q < NW; ++q) w[q] = agent_load(s + q);
#pragma unroll
    for (int q = 0; q < NW; ++q) ready = ready && (uint32_t)(w[q] >> 32) == epoch;
    if (ready) return true;
    if ((spin & 63u) == 0) {
      const long long now = wall_clock64();
      if (spin == 0) t0 = now;
      if (now - t0 > gs.limit || agent_load(gs.abort) != 0) {
        agent_store(gs.abort, 1);
        return false;
      }
    }
  }
}
__device__ inline double words_value(unsigned long long hi, unsigned long long lo) {
  return __longlong_as_double((long long)((hi << 32) | (lo & 0xffffffffull)));
}
__device__ inline unsigned long long value_word(double p, uint32_t epoch, bool low) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(p);
  return ((unsigned long long)epoch << 32) | (low ? (b & 0xffffffffull) : (b >> 32));
}

// Sum over all workgroups of the launch; false once the launch is aborted (the
// same answer for every thread of the workgroup).  sh: NV * (T / 64 + 1) + 1
// doubles.  With DRAIN the caller's stores are visible to every workgroup that
// returns; the barriers inside order the workgroup's LDS.
template <int NV, int T, bool DRAIN>
__device__ inline bool grid_sum(double (&v)[NV], const GridSlots& gs, uint32_t epoch, double* sh) {
  wg_partials<NV, T, DRAIN>(v, sh);
  double* res = sh + NV * (T / 64);
  if (threadIdx.x < 64) {
    wg_total<NV, T>(v, sh);
    const int lane = threadIdx.x;
    unsigned long long* mine = gs.words + (size_t)(2 * NV) * blockIdx.x;
    if (lane < 2 * NV) {
      double p = v[0];
#pragma unroll
      for (int q = 1; q < NV; ++q) p = (lane >> 1) == q ? v[q] : p;
      agent_store(mine + lane, value_word(p, epoch, lane & 1));
    }
    bool ok = true;
    double acc[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) acc[q] = 0;
    for (int g = lane; ok && g < gs.nwg; g += 64) {
      unsigned long long w[2 * NV];
      ok = poll_words<2 * NV>(gs.words + (size_t)(2 * NV) * g, epoch, gs, w);
#pragma unroll
      for (int q = 0; q < NV; ++q) acc[q] += words_value(w[2 * q], w[2 * q + 1]);
    }
    ok = __all(ok);
#pragma unroll
    for (int q = 0; q < NV; ++q) acc[q] = wave_sum(acc[q]);
    if (lane == 0) {
#pragma unroll
      for (int q = 0; q < NV; ++q) res[q] = acc[q];
      res[NV] = ok ? 1.0 : 0.0;
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] = res[q];
  return res[NV] != 0.0;
}

}  // namespace onsas
