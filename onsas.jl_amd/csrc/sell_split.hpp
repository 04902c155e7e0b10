// sell_split.hpp -- products with the sliced-ELL tangent for models whose slices
// do not fill the chip.  gfx950, wave64.
//
// One wave per slice runs a row's 15 or so rounds one after the other, each a
// column load and then the gathers it names; the waves of a large model hide one
// another's waits, but with fewer slices than about four a CU nothing else runs
// and a product is that chain (8 to 10 us where its bytes take 1 us).  Here four
// waves share a slice: wave w takes rounds w, w + 4, ..., kSplitPass of them with
// their columns, values and gathers in flight together, and the four sums of a
// row are added in wave order through LDS.  What the rows' epilogue needs, and
// the partial sums of the PCG's scalars, is loaded before the product.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "wave_ops.hpp"

namespace onsas {

constexpr int kSplitWaves = 4;  // waves per slice
constexpr int kSplitPass = 4;   // rounds in flight per wave (a row of 16 blocks: one pass)

// The rounds m, m + 4, ... of a pass (clamped to the last round; a slice without
// rounds, all its nodes outside every element, has nothing to load).
template <typename KT>
struct SplitPass {
  uint32_t j[kSplitPass];
  KT v[kSplitPass][9];
  __device__ inline void load(const int32_t* __restrict__ cp, const KT* __restrict__ vp, uint32_t rs,
                              int m, int rounds) {
#pragma unroll
    for (int q = 0; q < kSplitPass; ++q) {
      const uint32_t o = rs * (uint32_t)min(m + kSplitWaves * q, rounds - 1);
      j[q] = 3u * (uint32_t)cp[o];
#pragma unroll
      for (int e = 0; e < 9; ++e) v[q][e] = vp[9u * o + 64 * e];
    }
  }
  __device__ inline void add(const KT* __restrict__ x, int m, int rounds, KT (&a)[3]) const {
    KT xv[kSplitPass][3];
#pragma unroll
    for (int q = 0; q < kSplitPass; ++q)
#pragma unroll
      for (int c = 0; c < 3; ++c) xv[q][c] = x[j[q] + c];
#pragma unroll
    for (int q = 0; q < kSplitPass; ++q) {
      const bool ok = m + kSplitWaves * q < rounds;
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int d = 0; d < 3; ++d) a[c] += v[q][3 * c + d] * (ok ? xv[q][d] : KT(0));
    }
  }
};

// The sums of the slice's rows in wave 0 (lane = row); sh holds 9 x 64 values.
template <typename KT>
__device__ inline void split_combine(KT (&a)[3], KT* sh) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (w > 0)
#pragma unroll
    for (int c = 0; c < 3; ++c) sh[64 * (3 * (w - 1) + c) + lane] = a[c];
  __syncthreads();
  if (w == 0)
#pragma unroll
    for (int q = 0; q < kSplitWaves - 1; ++q)
#pragma unroll
      for (int c = 0; c < 3; ++c) a[c] += sh[64 * (3 * q + c) + lane];
}

// Sum of n partials by a 256-thread workgroup in two halves: the loads (4 a thread
// up to 1,024 partials) and, after other work, the sum: thread t adds entries t,
// t + 256, ..., then the wave, then the waves in order.  sh: 4 doubles.
struct PartSum {
  double a[4];
  __device__ inline void load(const double* __restrict__ p, int n) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = threadIdx.x + 256 * q;
      a[q] = i < n ? p[i] : 0.0;
    }
  }
  __device__ inline double wave_part(const double* __restrict__ p, int n) const {
    double s = ((a[0] + a[1]) + a[2]) + a[3];
    for (int i = threadIdx.x + 1024; i < n; i += 256) s += p[i];
    return wave_sum(s);
  }
};

}  // namespace onsas
