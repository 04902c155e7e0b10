// resident_solve.hip -- block-Jacobi PCG of small and mid-size models as one
// launch.  gfx950, wave64.
//
// The two-kernel iteration (k_pcg_A, k_pcg_B) of a model of a few thousand nodes
// is bound by kernel boundaries: 8.2 + 4.7 us of kernel time and 1.5 us of gaps
// an iteration at 1,680 nodes in FP32, where the bytes take 0.2 us.  Here the
// workgroups stay resident for the whole solve: the tangent rows live in
// registers (L lanes a row, NB blocks a lane), p, q, r, x and z of a row in its
// lanes, and an iteration costs two grid exchanges (grid_exchange.hpp), p.q and
// (r.z, r.r), with z handed over between them: 4.6 us at 1,680 nodes (27
// workgroups), 2.3 us at 125 nodes (one workgroup, z and the sums in LDS).
// The recurrences, the stop and breakdown rules and the scalars are those of
// k_pcg_A / k_pcg_B (p = z + beta p, q = K z + beta q); only the order of the
// sums differs.
#include <cstdlib>

#include "engine.hpp"
#include "grid_exchange.hpp"

namespace onsas {

namespace {

template <typename KT>
struct ResidentArgs {
  const int32_t* sell_ptr;
  const int32_t* slice_rounds;
  int64_t rstride;
  const int32_t* scol;
  const KT* sval;
  const KT* Dinv;
  const KT* r;
  KT* z;  // also hands z from workgroup to workgroup
  KT* x;
  const double* prz;
  const double* prr;
  int np;
  PcgState* st;
  unsigned long long* slots;  // 6 words per workgroup
  uint32_t base;              // epochs base + 1, base + 2, ... are new to the slots
  long long limit;
  int64_t nn;
};

// L lanes a block row (lane ph takes the row's slots ph, ph + L, ...: at most
// NB), T threads a workgroup.  Lanes 0, 1, 2 of a row hold the row's three
// components of every vector.  ONE: a single workgroup, z and the sums in LDS.
template <typename KT, int L, int NB, int T, bool ONE>
__global__ __launch_bounds__(T) void k_pcg_resident(ResidentArgs<KT> a) {
  __shared__ double shA[3 * (T / 64 + 1) + 1], shB[3 * (T / 64 + 1) + 1];
  __shared__ KT shz[ONE ? 3 * (T / L) : 1];
  const int t = threadIdx.x;
  const int ph = t % L;
  const int64_t i = ((int64_t)blockIdx.x * T + t) / L;
  const bool row = i < a.nn;
  const bool own = row && ph < 3;
  PcgState* st = a.st;
  const double tol2 = st->tol2;
  const int maxiter = st->maxiter;
  GridSlots gpq{a.slots, (int)gridDim.x, &st->aborted, a.limit};
  GridSlots gzr{a.slots + 2 * kMaxGridWg, (int)gridDim.x, &st->aborted, a.limit};

  KT v[NB][9];
  uint32_t cj[NB];  // byte offset of the column's z (a scalar base and 32-bit offsets)
  {
    const int64_t s = row ? i >> 6 : 0;
    const int32_t b0 = a.sell_ptr[s], rounds = a.slice_rounds[s];
    const int l = (int)(i & 63);
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int m = ph + L * q;
      const bool has = row && m < rounds;
      const int64_t b = b0 + a.rstride * (has ? m : 0);
      cj[q] = has ? 3u * (uint32_t)sizeof(KT) * (uint32_t)a.scol[b + l] : 0u;
#pragma unroll
      for (int e = 0; e < 9; ++e) v[q][e] = has ? a.sval[9 * b + 64 * e + l] : KT(0);
    }
  }
  KT xs = 0, rs = 0, zs = 0, ps = 0, qs = 0, d0 = 0, d1 = 0, d2 = 0;
  if (own) {
    xs = a.x[3 * i + ph];
    rs = a.r[3 * i + ph];
    zs = a.z[3 * i + ph];
    d0 = a.Dinv[9 * i + 3 * ph];
    d1 = a.Dinv[9 * i + 3 * ph + 1];
    d2 = a.Dinv[9 * i + 3 * ph + 2];
  }
  double zr[2] = {0, 0};
  for (int q = t; q < a.np; q += T) {
    zr[0] += a.prz[q];
    zr[1] += a.prr[q];
  }
  if (ONE && own) shz[3 * i + ph] = zs;
  wg_sum<2, T>(zr, shB);
  double rz = zr[0], rr = zr[1], rzp = 0;

  int k = 0, conv = 0, brk = 0;
  for (;; ++k) {
    conv = rr <= tol2;
    if (conv || k >= maxiter) break;
    KT zj[NB][3];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
#pragma unroll
      for (int c = 0; c < 3; ++c)
        zj[q][c] = ONE ? shz[cj[q] / sizeof(KT) + c]
                       : agent_load((const KT*)((const char*)a.z + cj[q]) + c);
    }
    KT a0 = 0, a1 = 0, a2 = 0;
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      a0 += v[q][0] * zj[q][0] + v[q][1] * zj[q][1] + v[q][2] * zj[q][2];
      a1 += v[q][3] * zj[q][0] + v[q][4] * zj[q][1] + v[q][5] * zj[q][2];
      a2 += v[q][6] * zj[q][0] + v[q][7] * zj[q][1] + v[q][8] * zj[q][2];
    }
    a0 = group_sum<L>(a0);
    a1 = group_sum<L>(a1);
    a2 = group_sum<L>(a2);
    double pq[1] = {0};
    if (own) {
      const KT beta = (KT)(k > 0 ? rz / rzp : 0.0);
      const KT ac = ph == 0 ? a0 : (ph == 1 ? a1 : a2);
      ps = zs + beta * ps;
      qs = ac + beta * qs;
      pq[0] = (double)ps * (double)qs;
    }
    if (ONE)
      wg_sum<1, T>(pq, shA);
    else if (!grid_sum<1, T, false>(pq, gpq, a.base + 1 + (uint32_t)k, shA))
      return;
    if (!(pq[0] > 0.0) || !isfinite(pq[0]) || !isfinite(rz)) {
      brk = 1;
      break;
    }
    const KT alpha = (KT)(rz / pq[0]);
    if (own) {
      xs += alpha * ps;
      rs -= alpha * qs;
    }
    const KT r0 = quad_lane<0>(rs), r1 = quad_lane<1>(rs), r2 = quad_lane<2>(rs);
    zr[0] = zr[1] = 0;
    if (own) {
      zs = d0 * r0 + d1 * r1 + d2 * r2;
      zr[0] = (double)rs * (double)zs;
      zr[1] = (double)rs * (double)rs;
      if (ONE)
        shz[3 * i + ph] = zs;
      else
        agent_store(a.z + 3 * i + ph, zs);
    }
    if (ONE)
      wg_sum<2, T>(zr, shB);
    else if (!grid_sum<2, T, true>(zr, gzr, a.base + 1 + (uint32_t)k, shB))
      return;
    rzp = rz;
    rz = zr[0];
    rr = zr[1];
  }
  if (own) a.x[3 * i + ph] = xs;
  if (blockIdx.x == 0 && t == 0) {
    st->rr_last = rr;
    st->k = k;
    if (brk) {
      st->breakdown = 1;
      st->breakdown_k = k;
    } else {
      st->done = 1;
      st->iters = k;
      st->converged = conv;
    }
  }
}

// L lanes a row: 4 for rows of up to 16 blocks (structured meshes: 15), 8 up to 32
inline int lanes_per_row(const Ctx* c) { return c->ell_width <= 16 ? 4 : 8; }
constexpr int kResidentBlocks = 4;  // blocks a lane keeps in registers
// Threads a workgroup: few, because a grid exchange waits for the workgroup's own
// barriers too.  A Newton solve of 1,680 / 1,728 / 4,913 nodes took 19.7 / 14.5 /
// 14.4 ms with 128 threads, 19.5 / 14.1 / 13.3 ms with 256 and 19.4 / 14.0 /
// 14.3 ms with 512 (FP64, 2,080 nodes: 5.0 / 4.7 / 5.0 ms), against 49.6 / 35.8 ms
// on two kernels an iteration: 256, and 512 where 256 would take more than
// kMaxGridWg workgroups.  The single workgroup gathers from LDS and takes as many
// threads as its registers allow (16 waves in FP32, 8 in FP64).
constexpr int kResidentThreads = 256;
constexpr int resident_one_threads(size_t kt) { return kt == 4 ? 1024 : 512; }

struct ResidentShape {
  int threads;
  int64_t grid;
};
inline ResidentShape resident_shape(const Ctx* c) {
  const int64_t lanes = c->nn * lanes_per_row(c);
  if (lanes <= resident_one_threads(c->kt)) return {resident_one_threads(c->kt), 1};
  int t = kResidentThreads;
  if ((lanes + t - 1) / t > kMaxGridWg) t *= 2;
  return {t, (lanes + t - 1) / t};
}

template <typename KT, int L>
void run_resident(Ctx* c, const ResidentArgs<KT>& a, const ResidentShape& sh) {
  constexpr int T1 = resident_one_threads(sizeof(KT)), T = kResidentThreads;
  const dim3 grid((unsigned)sh.grid);
  if (sh.grid == 1)
    hipLaunchKernelGGL((k_pcg_resident<KT, L, kResidentBlocks, T1, true>), grid, dim3(T1), 0,
                       c->stream, a);
  else if (sh.threads == T)
    hipLaunchKernelGGL((k_pcg_resident<KT, L, kResidentBlocks, T, false>), grid, dim3(T), 0,
                       c->stream, a);
  else
    hipLaunchKernelGGL((k_pcg_resident<KT, L, kResidentBlocks, 2 * T, false>), grid, dim3(2 * T), 0,
                       c->stream, a);
}

template <typename KT>
int resident_t(Ctx* c) {
  ResidentArgs<KT> a{};
  a.sell_ptr = c->d_sell_ptr;
  a.slice_rounds = c->d_slice_rounds;
  a.rstride = c->ell_rounds ? 64 * c->nslices : 64;
  a.scol = c->d_sell_col;
  a.sval = (const KT*)c->d_Ksell;
  a.Dinv = (const KT*)c->d_Dinv;
  a.r = (const KT*)c->d_pr;
  a.z = (KT*)c->d_pz;
  a.x = (KT*)c->d_px;
  a.prz = part(c, kPartRZ0);
  a.prr = part(c, kPartRR);
  a.np = c->np;
  a.st = &c->d_sc->pcg;
  a.slots = c->d_gslots;
  a.base = c->gslot_epoch;
  a.limit = c->gslot_ticks;
  a.nn = c->nn;
  const ResidentShape sh = resident_shape(c);
  if (lanes_per_row(c) == 4)
    run_resident<KT, 4>(c, a, sh);
  else
    run_resident<KT, 8>(c, a, sh);
  ONSAS_HIP_TRY(c, hipGetLastError());
  return ONSAS_OK;
}

}  // namespace

// Whether a block-Jacobi PCG of this model runs as one launch: rows short enough
// for the lanes' registers and a grid of at most kMaxGridWg workgroups (16,384
// rows of up to 16 blocks, 8,192 of up to 32).
bool pcg_resident_fits(const Ctx* c) {
  return kSellLanes == 1 && c->ell_width <= 8 * kResidentBlocks &&
         resident_shape(c).grid <= kMaxGridWg;
}

int pcg_resident_alloc(Ctx* c) {
  const char* e = std::getenv("ONSAS_PCG_RESIDENT");
  c->pcg_resident = pcg_resident_fits(c) && !(e && e[0] == '0');
  if (const char* t = std::getenv("ONSAS_RESIDENT_TICKS")) c->gslot_ticks = std::atoll(t);
  if (!c->pcg_resident) return ONSAS_OK;
  const size_t words = 6 * (size_t)kMaxGridWg * sizeof(unsigned long long);
  ONSAS_HIP_TRY(c, hipMalloc((void**)&c->d_gslots, words));
  ONSAS_HIP_TRY(c, hipMemsetAsync(c->d_gslots, 0, words, c->stream));
  return ONSAS_OK;
}

int launch_pcg_resident(Ctx* c) {
  if (c->gslot_epoch > 0xf0000000u) {  // the epochs wrap: clear the slots' marks
    ONSAS_HIP_TRY(c, hipMemsetAsync(c->d_gslots, 0,
                                    6 * (size_t)kMaxGridWg * sizeof(unsigned long long), c->stream));
    c->gslot_epoch = 1;
  }
  return c->precision == ONSAS_PRECISION_FP64 ? resident_t<double>(c) : resident_t<float>(c);
}

}  // namespace onsas
