// grid_exchange.hpp -- sums and vectors shared by the workgroups of one resident
// launch (the solver kernels that run a whole solve in one launch).  gfx950.
//
// Every workgroup of such a launch is resident at once (the host holds the grid to what
// the device reports for the kernel: resident_rule.hpp), so workgroups may wait for one
// another.  A grid-wide
// sum is one exchange: each workgroup writes its partial into its own slot and
// polls the slots of all others.  The slot words are 8 bytes, (epoch << 32) |
// half of the double, so a word carries its own "ready" mark and the sum is
// exact; the partials are added by a fixed tree, the same in every workgroup,
// so all of them take the same branches and a solve is bit-identical from run
// to run, in either meeting place, as long as no wait expires (the general kernels
// add in another order).  A sum alone, measured on one MI355X: 1.2 us for 2 workgroups, 1.9 us for
// 32, 2.4 us for 64 and 3.3 us for 128 across the device, against 4 to 8 us for a
// kernel boundary with its drain, launch and first loads.  Vectors are handed over a
// node at a time with a mark of their own (share_node), so nothing else orders the
// workgroups' memory and the read-only data stays cached.
//
// Waits are bounded: a workgroup that polls past `limit` clock ticks (or sees
// another's abort) raises the abort word and the launch drains; the host then takes the
// solve again across the device, or on the general kernels, and comes back to the fastest
// path some solves later.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "share_mark.hpp"
#include "wave_ops.hpp"

namespace onsas {

constexpr int kMaxGridWg = 128;  // workgroups of a resident launch
constexpr int kPollSlots = 64;   // slots that grid_sum4 polls at a time
constexpr size_t kGridSlotWords = 32 * kMaxGridWg;  // the PCG's slots: sums of four values, four times

template <typename T>
__device__ inline T agent_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ inline void agent_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Where the workgroups meet.  Device: the loads and stores of everything shared pass
// the caches (sc1).  One XCD: they meet in its L2 (stores are written through to it,
// loads take sc0 nt and so do not stay in the CU's cache); an exchange of 27 / 64
// workgroups is 1.1 / 1.1 us against 1.9 / 2.4.  A load that did come from the CU's
// cache would show an old mark and be repeated.
enum class Meet { kDevice, kXcd };

// 16 bytes that other workgroups write; the caller keeps the load in its loop (poll).
using SharedBuf = __amdgpu_buffer_rsrc_t;
__device__ inline SharedBuf shared_buf(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
template <Meet M>
constexpr int kSharedLoad = M == Meet::kXcd ? 3 : 16;  // sc0 nt, sc1
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <Meet M>
__device__ inline u32x4 shared_load(SharedBuf b, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(b, off, 0, kSharedLoad<M>);
}
template <Meet M>
__device__ inline void shared_store(unsigned long long* p, unsigned long long w) {
  if (M == Meet::kXcd)
    __hip_atomic_store(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  else
    agent_store(p, w);
}
// the XCD this wave runs on
__device__ inline int xcd_id() {
  int x;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(x));
  return x;
}

struct GridSlots {
  unsigned long long* words;  // kMaxGridWg slots
  int nwg, id;
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

// load() until it says that everything has arrived; false once the launch is aborted
template <typename Load>
__device__ inline bool poll(const GridSlots& gs, Load load) {
  long long t0 = 0;
  for (uint32_t spin = 0;; ++spin) {
    asm volatile("" ::: "memory");  // the loads stay in the loop
    if (load()) return true;
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
// N values at the byte offsets off, a high and a low word each, once all carry the epoch
template <Meet M, int N>
__device__ inline bool poll_values(SharedBuf buf, const uint32_t (&off)[N], uint32_t epoch,
                                   const GridSlots& gs, double (&v)[N]) {
  return poll(gs, [&] {
    u32x4 w[N];
    bool ready = true;
#pragma unroll
    for (int q = 0; q < N; ++q) w[q] = shared_load<M>(buf, off[q]);
#pragma unroll
    for (int q = 0; q < N; ++q) {
      ready = ready && w[q][1] == epoch && w[q][3] == epoch;
      v[q] = __hiloint2double((int)w[q][0], (int)w[q][2]);
    }
    return ready;
  });
}
__device__ inline unsigned long long value_word(double p, uint32_t epoch, bool low) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(p);
  return ((unsigned long long)epoch << 32) | (low ? (b & 0xffffffffull) : (b >> 32));
}

// A node of a vector that its neighbours read: 16 bytes, its three components and a
// mark (FP64: twice 16 bytes, each with 12 bytes of the components and a mark).  No
// memory model says that an aligned 16-byte store or load of a lane is seen whole; it is
// one request to one cache line, and no mixture has been seen.  The mark does not rest on
// that: it is made of the epoch and the other three words (share_mark.hpp).  Against the
// epoch alone that is 2 % of an FP64 solve of 2,080 nodes and nothing in FP32; a test of
// one word after the other under branches took 10 % of it.  A sum between the readers' use and the next hand-over makes sure
// that nothing is overwritten before all have read it.
template <typename KT>
constexpr uint32_t kShareBytes = 4 * sizeof(KT);  // per node
template <typename KT>
constexpr int kShareLanes = sizeof(KT) / 4;       // lanes that store a node
template <Meet M>
__device__ inline void shared_store(SharedBuf b, uint32_t off, u32x4 w) {
  if (M == Meet::kXcd)
    __builtin_amdgcn_raw_buffer_store_b128(w, b, off, 0, 1);   // sc0
  else
    __builtin_amdgcn_raw_buffer_store_b128(w, b, off, 0, 16);  // sc1
}
// node i's part of lane `part` (0, and in FP64 0 and 1)
template <Meet M>
__device__ inline void share_node(SharedBuf z, uint32_t i, int part, float a, float b, float c,
                                  uint32_t epoch) {
  (void)part;
  const uint32_t x = __float_as_uint(a), y = __float_as_uint(b), w = __float_as_uint(c);
  shared_store<M>(z, kShareBytes<float> * i, u32x4{x, y, w, share_mark(x, y, w, epoch)});
}
template <Meet M>
__device__ inline void share_node(SharedBuf z, uint32_t i, int part, double a, double b, double c,
                                  uint32_t epoch) {
  const double x = part ? c : a;
  const uint32_t l = (uint32_t)__double2loint(x), h = (uint32_t)__double2hiint(x),
                 o = (uint32_t)(part ? __double2hiint(b) : __double2loint(b));
  shared_store<M>(z, kShareBytes<double> * i + 16u * part,
                  u32x4{l, h, o, share_mark(l, h, o, epoch)});
}
// The three components of the nodes at the byte offsets off, once they carry the
// epoch; false once the launch is aborted.
template <Meet M, typename KT, int N>
__device__ inline bool gather_shared(SharedBuf z, const uint32_t (&off)[N], uint32_t epoch,
                                     const GridSlots& gs, KT (&zj)[N][3]) {
  constexpr int P = kShareLanes<KT>;
  return poll(gs, [&] {
    u32x4 w[N][P];
    uint32_t off_mark = 0;  // zero once every mark is the epoch's (no branch a word)
#pragma unroll
    for (int q = 0; q < N; ++q)
#pragma unroll
      for (int p = 0; p < P; ++p) w[q][p] = shared_load<M>(z, off[q] + 16u * p);
#pragma unroll
    for (int q = 0; q < N; ++q) {
#pragma unroll
      for (int p = 0; p < P; ++p)
        off_mark |= w[q][p][3] ^ share_mark(w[q][p][0], w[q][p][1], w[q][p][2], epoch);
      if constexpr (P == 1) {
#pragma unroll
        for (int c = 0; c < 3; ++c) zj[q][c] = __uint_as_float(w[q][0][c]);
      } else {
        zj[q][0] = __hiloint2double((int)w[q][0][1], (int)w[q][0][0]);
        zj[q][1] = __hiloint2double((int)w[q][1][2], (int)w[q][0][2]);
        zj[q][2] = __hiloint2double((int)w[q][1][1], (int)w[q][1][0]);
      }
    }
    return off_mark == 0;
  });
}

// The four sums over all workgroups of the launch; false once the launch is
// aborted (the same answer for every thread of the workgroup).  sh: 4 T / 64 + 5
// doubles, free again at the caller's next barrier.  late: an LDS word that a thread
// has set whose own wait expired before the sum; nothing is published then.  A load
// takes 16 slots (a lane its sum's 16 bytes of one).
template <Meet M, int T>
__device__ inline bool grid_sum4(double (&v)[4], const GridSlots& gs, uint32_t epoch, double* sh,
                                 const int* late) {
  double* res = sh + 4 * (T / 64);
  const int lane = threadIdx.x & 63;
  {
    const double p = wave_sum4(v);
    if (lane < 4) sh[4 * (threadIdx.x >> 6) + lane] = p;
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const double p = wg_sum4<T>(sh);
    bool ok = *late == 0;
    if (ok && lane < 4) {
      unsigned long long* mine = gs.words + 8 * (size_t)gs.id + 2 * lane;
      shared_store<M>(mine, value_word(p, epoch, false));
      shared_store<M>(mine + 1, value_word(p, epoch, true));
    }
    const SharedBuf buf = shared_buf(gs.words, 64u * kMaxGridWg);
    double acc = 0;
    for (int g0 = 0; ok && g0 < gs.nwg; g0 += kPollSlots) {
      double x[4];
      uint32_t off[4];
      bool has[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int g = g0 + 16 * j + (lane >> 2);
        has[j] = g < gs.nwg;
        off[j] = 64u * (has[j] ? g : gs.id) + 16u * (lane & 3);
      }
      ok = poll_values<M, 4>(buf, off, epoch, gs, x);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc += has[j] ? x[j] : 0.0;
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
