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
// to run.  A sum alone, measured on one MI355X: 1.2 us for 1 to 8 workgroups, 2.0 us for 32,
// 3.3 us for 128, against 4 to 8 us for a kernel boundary with its drain,
// launch and first loads.
//
// Everything shared goes through device-scope loads and stores (they bypass the
// per-XCD L2s), and a workgroup's vector stores are complete (vmcnt 0, then the
// barrier, in grid_sum4) before its partial is published, so no L2
// write-back or invalidation is needed and the read-only data stays cached.
// Waits are bounded: a workgroup that polls past `limit` clock ticks (or sees
// another's abort) raises the abort word and the launch drains; the host then
// solves with the one-kernel-per-step path.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "wave_ops.hpp"

namespace onsas {

constexpr int kMaxGridWg = 128;  // workgroups of a resident launch
constexpr int kPollSlots = 64;   // slots that grid_sum4 polls at a time
constexpr size_t kGridSlotWords = 16 * kMaxGridWg;  // the PCG's slots: sums of four values, twice

template <typename T>
__device__ inline T agent_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ inline void agent_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The loads of values that other workgroups write: past the caches like
// agent_load, and 12 or 16 bytes an instruction.  Every value among them is at
// most 8 bytes and aligned, and carries its own mark.
using SharedBuf = __amdgpu_buffer_rsrc_t;
__device__ inline SharedBuf shared_buf(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
constexpr int kSharedLoad = (int)(0x80000000u | 16u);  // volatile (each poll loads anew), sc1
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ inline void shared_load3(SharedBuf b, uint32_t off, uint32_t (&w)[3]) {
  const u32x3 v = __builtin_amdgcn_raw_buffer_load_b96(b, off, 0, kSharedLoad);
  w[0] = v[0];
  w[1] = v[1];
  w[2] = v[2];
}
__device__ inline void shared_load2(SharedBuf b, uint32_t off, unsigned long long (&w)[2]) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(b, off, 0, kSharedLoad);
  w[0] = ((unsigned long long)v[1] << 32) | v[0];
  w[1] = ((unsigned long long)v[3] << 32) | v[2];
}
__device__ inline void shared_load3(SharedBuf b, uint32_t off, unsigned long long (&w)[3]) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(b, off, 0, kSharedLoad);
  const u32x2 u = __builtin_amdgcn_raw_buffer_load_b64(b, off + 16, 0, kSharedLoad);
  w[0] = ((unsigned long long)v[1] << 32) | v[0];
  w[1] = ((unsigned long long)v[3] << 32) | v[2];
  w[2] = ((unsigned long long)u[1] << 32) | u[0];
}
// this wave's stores have reached the device-coherent level
__device__ inline void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

struct GridSlots {
  unsigned long long* words;  // kMaxGridWg slots of the sum's 2 NV words each
  int nwg;
  int* abort;                 // device word: nonzero once a wait has expired
  long long limit;            // ticks of the 100 MHz clock a wait may take
};

// Four sums over the workgroup at once, lane l of a wave holding a part of sum
// l & 3 from the first step on, so that a tree step is one addition and not four.
// First: the wave's part of sum l & 3, in every lane (v: the thread's parts, all
// 64 lanes active).
__device__ inline double wave_sum4(const double (&v)[4]) {
  const int q = threadIdx.x & 3;
  const double a = group_sum<4>(v[0]), b = group_sum<4>(v[1]), c = group_sum<4>(v[2]),
               d = group_sum<4>(v[3]);
  return stride_sum<4>((q & 2) ? ((q & 1) ? d : c) : ((q & 1) ? b : a));
}
// Then, past a barrier, the workgroup's sum l & 3 from the waves' parts in sh (T threads).
template <int T>
__device__ inline double wg_sum4(const double* sh) {
  static_assert(4 * (T / 64) <= 64, "a part per lane");
  const int lane = threadIdx.x & 63;
  return stride_sum<4>(lane < 4 * (T / 64) ? sh[lane] : 0.0);
}

// N values at the byte offsets off, two words each, once all of them carry the
// epoch; false once the launch is aborted.
template <int N>
__device__ inline bool poll_values(SharedBuf buf, const uint32_t (&off)[N], uint32_t epoch,
                                   const GridSlots& gs, unsigned long long (&w)[N][2]) {
  long long t0 = 0;
  for (uint32_t spin = 0;; ++spin) {
    bool ready = true;
#pragma unroll
    for (int q = 0; q < N; ++q) shared_load2(buf, off[q], w[q]);
#pragma unroll
    for (int q = 0; q < N; ++q)
      ready = ready && (uint32_t)(w[q][0] >> 32) == epoch && (uint32_t)(w[q][1] >> 32) == epoch;
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

// The four sums over all workgroups of the launch; false once the launch is
// aborted (the same answer for every thread of the workgroup).  sh: 4 T / 64 + 5
// doubles, free again at the caller's next barrier.  The stores that the caller
// made before it are complete at the device-coherent level before its part is
// published.  late: an LDS word that a thread has set whose own wait expired
// before the sum; nothing is published then.  A load takes 16 slots (a lane its
// sum's 16 bytes of one).
template <int T>
__device__ inline bool grid_sum4(double (&v)[4], const GridSlots& gs, uint32_t epoch, double* sh,
                                 const int* late) {
  double* res = sh + 4 * (T / 64);
  const int lane = threadIdx.x & 63;
  {
    const double p = wave_sum4(v);
    if (lane < 4) sh[4 * (threadIdx.x >> 6) + lane] = p;
  }
  stores_done();
  __syncthreads();
  if (threadIdx.x < 64) {
    const double p = wg_sum4<T>(sh);
    bool ok = *late == 0;
    if (ok && lane < 4) {
      unsigned long long* mine = gs.words + 8 * (size_t)blockIdx.x + 2 * lane;
      agent_store(mine, value_word(p, epoch, false));
      agent_store(mine + 1, value_word(p, epoch, true));
    }
    const SharedBuf buf = shared_buf(gs.words, 64u * kMaxGridWg);
    double acc = 0;
    for (int g0 = 0; ok && g0 < gs.nwg; g0 += kPollSlots) {
      unsigned long long w[4][2];
      uint32_t off[4];
      bool has[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int g = g0 + 16 * j + (lane >> 2);
        has[j] = g < gs.nwg;
        off[j] = 64u * (has[j] ? g : blockIdx.x) + 16u * (lane & 3);
      }
      ok = poll_values<4>(buf, off, epoch, gs, w);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc += has[j] ? words_value(w[j][0], w[j][1]) : 0.0;
    }
    ok = __all(ok);
    acc = stride_sum<4>(acc);
    if (lane < 4) res[lane] = acc;
    if (lane == 0) res[4] = ok ? 1.0 : 0.0;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = res[q];
  return res[4] != 0.0;
}

}  // namespace onsas
