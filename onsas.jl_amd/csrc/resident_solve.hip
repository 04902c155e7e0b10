// resident_solve.hip -- block-Jacobi PCG and GMRES of small and mid-size models,
// each solve one launch.  gfx950, wave64.
//
// PCG.
// The two-kernel iteration (k_pcg_A, k_pcg_B) of a model of a few thousand nodes
// is bound by kernel boundaries: 8.2 + 4.7 us of kernel time and 1.5 us of gaps
// an iteration at 1,680 nodes in FP32, where the bytes take 0.2 us.  Here the
// workgroups stay resident for the whole solve: the tangent rows live in
// registers (L lanes a row, NB blocks a lane), p, q, r, x and z of a row in its
// lanes.  What is left is the latency of one workgroup hearing from the others,
// so an iteration does it twice only, once for the neighbours' z and once for one
// sum of four values (grid_exchange.hpp), as in the single-reduction form of the
// method (A. T. Chronopoulos and C. W. Gear, J. Comput. Appl. Math. 25, 1989):
//   w = K z;  r.z, r.r, z.w and z.q + p.w, with p and q of the iteration before
//   p <- z + beta p, q <- w + beta q;  p.q <- z.w + beta (z.q + p.w) + beta^2 p.q
// The last line is p.q written out (no conjugacy is assumed), so the recurrences and
// the stop and breakdown rules are those of k_pcg_A / k_pcg_B.  It does not see the
// rounding of p and q and hands its error on, times beta^2: an error estimate goes
// with it (kPqError), and p.q is summed from p and q where that has grown, and before
// every breakdown.  z needs no sum to be safe to read: a node that
// is not there yet carries an old epoch.
// An iteration takes 2.4 us at 1,680 nodes (27 workgroups, met in one XCD; FP64 2.7 us),
// 1.0 us at 125 nodes (one workgroup, z and the sums in LDS; FP64 1.2 us).  Met in device
// memory it is 3.4 us; with p.q and (r.z, r.r) as two sums, z safe to read only after the
// second, a tree per sum and 4- and 8-byte loads it was 4.6 and 2.6 us.  A pipelined
// recurrence (P. Ghysels and W. Vanroose, Parallel Comput. 40, 2014) would hide the sum
// behind the product, but loses the residual: on the host, for a 13 x 9 x 11 box, it
// stalls at a true residual of 2.5e-2 in FP32 (1e-5 here, rtol 1e-6) and takes 409 for 314
// iterations to 2e-10 for 8e-13 in FP64 (rtol 1e-12); the residual computed anew every 50
// iterations mends FP64 and not FP32.  Polling by every wave of a
// workgroup instead of one costs 1 us.
#include <unistd.h>

#include <atomic>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <type_traits>

#include <hip/hip_ext.h>

#include "engine.hpp"
#include "grid_exchange.hpp"
#include "resident_rule.hpp"

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
  const uint8_t* mask;
  const double* b;     // right-hand side; of a Newton step f_ext
  KT* x;
  unsigned long long* z;  // z, handed from workgroup to workgroup (share_node)
  Scalars* sc;         // device: the abort word, a Newton step's norms
  Scalars* host;       // pinned host: the results
  unsigned long long* slots;  // four regions of 8 words per workgroup
  uint32_t base;              // epochs base + 1, base + 2, ... are new to the slots and z
  int nwg, xcd;               // workgroups; of kXcd launches every 8th, from xcd on
  long long limit;
  int64_t nn;
  int maxiter;
  InnerTol tol;
  // a Newton step (fint not null)
  const double* fint;
  const KT* x0;        // warm start or null
  KT* warm;            // takes a copy of x, or null
  double *res, *U;
};

// The estimate of p.q's error is 2 u (z.w + |beta (z.q + p.w)| + beta^2 p.q), u the unit
// of KT, and beta^2 times the estimate before; past kPqError u p.q a sum of its own takes
// the place of the recurrence (an exchange: 2 of the 225 iterations of a 13 x 9 x 11 box,
// none of 69 at 4 x 4 x 4, every 30th on a flat box, every 5th to 16th where stiffnesses
// spread over two to seven decades).  Of chains of 20 bars over 2 / 4 / 6 / 7 decades in
// FP32 (a host model, 192 each) the largest error of p.q is then 29 / 100 / 480 / 1,100 u,
// and the iterations are the direct sum's within 2 %; without it 67 / 7,200 / 3e5 / 5e7 u,
// up to a quarter more iterations, and breakdowns of definite tangents.  With 64 u 6 / 32 /
// 210 / 670 u for about twice as many sums.  The estimate is made beside the division that
// alpha waits for; it and its sums take 1 to 3 % of the solves' time, a fifth sum in every
// exchange took 8 to 10 %.
constexpr double kPqError = 256;
template <typename KT>
constexpr double kUnit = sizeof(KT) == 4 ? 0x1p-24 : 0x1p-53;

// PcgState::aborted of a launch whose workgroups did not share one XCD
constexpr int kNotOneXcd = 2;

// a result for the host, in pinned host memory
template <typename T>
__device__ inline void host_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// L lanes a block row (lane ph takes the row's slots ph, ph + L, ...: at most
// NB), T threads a workgroup.  Lanes 0, 1, 2 of a row hold the row's three
// components of every vector.  ONE: a single workgroup, z and the sums in LDS.
//
// The launch starts from the right-hand side and ends with the results in pinned
// host memory; of a Newton step it is all that follows the assembly: residual,
// warm start, stopping tolerance, solve, update of U and norms (k_residual,
// k_spmv_sell, k_warm_dots, k_warm_init, k_pcg_init_finalize, k_update and
// k_finalize_newton of the general path, with two copies to the host and one on
// the device: some 60 us of a step of 195 us at 125 nodes, now 5 us; the step 195 ->
// 152 us, and 143 us since the assembly stamps its own events).
//
// The sums take two slot regions in turn: a workgroup may be in sum k + 1 while
// another still reads sum k.  z has one buffer: the sum before its next hand-over is
// complete only when every workgroup has made its product.
//
// kXcd: every 8th workgroup takes part, from the context's own first one on (contexts
// that solve at the same time would hold each other's places on a shared XCD).  Consecutive workgroups go round the 8 XCDs, so
// these share one, which a first sum across the device confirms (if not, nothing has
// been done and the host launches the other kernel); they then meet in its L2.
template <typename KT, int L, int NB, int T, bool ONE, Meet M>
__global__ __launch_bounds__(T) void k_pcg_resident(ResidentArgs<KT> a) {
  constexpr int kSpread = M == Meet::kXcd ? 8 : 1;
  if (M == Meet::kXcd && (int)(blockIdx.x % kSpread) != a.xcd) return;
  const int wg = (int)(blockIdx.x / kSpread);
  __shared__ double sh[4 * (T / 64) + 5];
  __shared__ __align__(16) KT shz[ONE ? 4 * (T / L) : 4];  // a node's z and a pad: 16-byte reads
  __shared__ int late;  // a wait for z has expired
  const int t = threadIdx.x;
  const int ph = t % L;
  const int64_t i = ((int64_t)wg * T + t) / L;
  const bool row = i < a.nn;
  const bool own = row && ph < 3;
  uint32_t ep = a.base;
  GridSlots gs{a.slots, a.nwg, wg, &a.sc->pcg.aborted, a.limit};
  // the four sums over the launch; false (and *host says so) once it is aborted
  auto sums = [&](double(&s)[4], auto m) -> bool {
    constexpr Meet W = decltype(m)::value;
    ++ep;
    if (ONE) {
      const double p = wave_sum4(s);
      if ((t & 63) < 4) sh[4 * (t >> 6) + (t & 63)] = p;
      __syncthreads();
      const double q4 = wg_sum4<T>(sh);
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q] = read_lane(q4, q);
      return true;
    }
    gs.words = a.slots + ((ep & 1u) + (W == Meet::kXcd ? 2u : 0u)) * (8 * kMaxGridWg);
    if (grid_sum4<W, T>(s, gs, ep, sh, &late)) return true;
    if (t == 0) host_store(&a.host->pcg.aborted, 1);
    return false;
  };

  KT v[NB][9];
  uint32_t cj[NB];  // the column's z: its byte offset, or its index in shz
  {
    const int64_t s = row ? i >> 6 : 0;
    const int32_t b0 = a.sell_ptr[s], rounds = a.slice_rounds[s];
    const int l = (int)(i & 63);
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int m = ph + L * q;
      const bool has = row && m < rounds;
      const int64_t b = b0 + a.rstride * (has ? m : 0);
      cj[q] = (ONE ? 4u : kShareBytes<KT>) * (uint32_t)(has ? a.scol[b + l] : 0);
#pragma unroll
      for (int e = 0; e < 9; ++e) v[q][e] = has ? a.sval[9 * b + 64 * e + l] : KT(0);
    }
  }
  // w = K z of the row's component ph from the columns' z
  auto product = [&](const KT(&zj)[NB][3]) -> KT {
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
    return ph == 0 ? a0 : (ph == 1 ? a1 : a2);
  };
  const int64_t dof = 3 * i + ph;
  const bool newton = a.fint != nullptr;
  // read before the first sum: the first workgroup overwrites it as early as after a
  // breakdown in iteration 0
  double before_b2 = read_lane(a.tol.forcing ? a.sc->nwt.prev_b2 : 0.0, 0);
  asm volatile("" : "+s"(before_b2));
  KT xs = 0, rs = 0, zs = 0, ps = 0, qs = 0, d0 = 0, d1 = 0, d2 = 0, bk = 0;
  double u = 0, sm[4] = {0, 0, 0, 0};
  bool freed = false;
  if (own) {
    freed = !((a.mask[i] >> ph) & 1u);
    d0 = a.Dinv[9 * i + 3 * ph];
    d1 = a.Dinv[9 * i + 3 * ph + 1];
    d2 = a.Dinv[9 * i + 3 * ph + 2];
    const double be = a.b[dof];
    double r = be;
    if (newton) {
      u = a.U[dof];
      r -= a.fint[dof];
      sm[1] = be * be;
    }
    if (!freed) r = 0;
    if (newton) {
      a.res[dof] = r;
      sm[0] = r * r;
    }
    bk = (KT)r;
  }
  const std::integral_constant<Meet, M> here;
  if (M == Meet::kXcd) {  // do they share one XCD?  n sum x^2 = (sum x)^2
    if (t == 0) late = 0;
    __syncthreads();
    const double x = t == 0 ? (double)xcd_id() : 0.0;
    double q[4] = {x, x * x, 0, 0};
    if (!sums(q, std::integral_constant<Meet, Meet::kDevice>())) return;
    if (a.nwg * q[1] != q[0] * q[0]) {
      if (t == 0) host_store(&a.host->pcg.aborted, kNotOneXcd);
      return;
    }
  }
  // warm start: x = al x0, r = b - al t with t = K x0 and al = t.b / t.t, the scale
  // that minimises ||b - al t|| (as k_warm_init)
  KT x0 = 0, tw = 0;
  if (a.x0) {
    KT xj[NB][3];
#pragma unroll
    for (int q = 0; q < NB; ++q)
#pragma unroll
      for (int c = 0; c < 3; ++c)
        xj[q][c] = a.x0[cj[q] / (ONE ? 4u : kShareBytes<KT>) * 3 + c];
    tw = product(xj);
    if (own && freed) {
      x0 = a.x0[dof];
      sm[2] = (double)tw * (double)bk;
      sm[3] = (double)tw * (double)tw;
    }
  }
  if (t == 0) late = 0;
  __syncthreads();
  if (!sums(sm, here)) return;
  const double r2 = sm[0], f2 = sm[1];
  const double al = a.x0 && sm[3] > 0 && isfinite(sm[2]) && isfinite(sm[3]) ? sm[2] / sm[3] : 0.0;
  if (own) {
    xs = freed ? (KT)(al * (double)x0) : KT(0);
    rs = freed ? (a.x0 ? (KT)((double)bk - al * (double)tw) : bk) : KT(0);
  }
  const SharedBuf z = shared_buf(a.z, kShareBytes<KT> * (uint32_t)a.nn);
  // z = D^-1 r, published
  auto next_z = [&]() {
    const KT r0 = quad_lane<0>(rs), r1 = quad_lane<1>(rs), rz2 = quad_lane<2>(rs);
    if (own) zs = d0 * r0 + d1 * r1 + d2 * rz2;
    if (ONE) {
      if (own) shz[4 * i + ph] = zs;
      __syncthreads();
    } else {
      const KT s0 = quad_lane<0>(zs), s1 = quad_lane<1>(zs), s2 = quad_lane<2>(zs);
      if (row && ph < kShareLanes<KT>) share_node<M>(z, (uint32_t)i, ph, s0, s1, s2, ep);
    }
  };
  next_z();

  double rz = 0, rr = 0, rzp = 0, pq = 0, pqe = 0, bb = 0, eta = 0, tol2 = 0;
  int k = 0, conv = 0, brk = 0;
  for (;; ++k) {
    KT zj[NB][3];
    if (ONE) {
#pragma unroll
      for (int q = 0; q < NB; ++q)
#pragma unroll
        for (int c = 0; c < 3; ++c) zj[q][c] = shz[cj[q] + c];
    } else if (!gather_shared<M, KT, NB>(z, cj, ep, gs, zj)) {
      late = 1;
    }
    const KT w = product(zj);
    sm[0] = sm[1] = sm[2] = sm[3] = 0;
    if (own) {
      sm[0] = (double)rs * (double)zs;
      sm[1] = (double)rs * (double)rs;
      sm[2] = (double)zs * (double)w;
      sm[3] = k > 0 ? (double)zs * (double)qs + (double)ps * (double)w : (double)bk * (double)bk;
    }
    if (!sums(sm, here)) return;
    if (k == 0) {
      bb = sm[3];
      sm[3] = 0;
      eta = inner_eta(a.tol, bb, f2, before_b2);
      tol2 = eta * eta * bb;
    }
    rzp = rz;
    rz = sm[0];
    rr = sm[1];
    conv = rr <= tol2;
    if (conv || k >= a.maxiter) break;
    const KT beta = (KT)(k > 0 ? rz / rzp : 0.0);
    const double bt = (double)beta, b2 = bt * bt, b2pq = b2 * pq;
    pq = sm[2] + (bt * sm[3] + b2pq);
    KT alpha = (KT)(rz / pq);
    pqe = b2 * pqe + 2 * kUnit<KT> * (fabs(sm[2]) + fabs(bt * sm[3]) + b2pq);
    if (own) {
      ps = zs + beta * ps;
      qs = w + beta * qs;
    }
    // (the same answer in every workgroup; pq > 0 otherwise)
    if (!(pqe <= kPqError * kUnit<KT> * pq) || !isfinite(pq) || !isfinite(rz)) {
      sm[0] = own ? (double)ps * (double)qs : 0.0;
      sm[1] = sm[2] = sm[3] = 0;
      if (ONE) __syncthreads();  // the last sums have been read
      if (!sums(sm, here)) return;
      pq = sm[0];
      pqe = 0;
      if (!(pq > 0.0) || !isfinite(pq) || !isfinite(rz)) {
        brk = 1;
        break;
      }
      alpha = (KT)(rz / pq);
    }
    if (own) {
      xs += alpha * ps;
      rs -= alpha * qs;
    }
    next_z();
  }
  if (own) a.x[dof] = xs;
  // Newton update: U[free] += x, with the norms of x and of U before
  double du = 0;
  sm[0] = sm[1] = sm[2] = sm[3] = 0;
  if (newton && !brk) {
    if (own) {
      du = freed ? (double)xs : 0.0;
      sm[0] = du * du;
      sm[1] = u * u;
    }
    if (ONE) __syncthreads();  // the last sums have been read
    if (!sums(sm, here)) return;
    if (own) {
      a.U[dof] = u + du;
      if (a.warm) a.warm[dof] = xs;
    }
  }
  if (wg == 0 && t == 0) {
    PcgState* st = &a.host->pcg;
    host_store(&st->bb, bb);
    host_store(&st->rr_last, rr);
    host_store(&st->k, (int32_t)(ep - a.base));  // epochs used
    host_store(&st->breakdown, brk);
    host_store(&st->breakdown_k, brk ? k : -1);
    host_store(&st->iters, k);
    host_store(&st->converged, brk ? 0 : conv);
    host_store(&st->done, 1);
    if (newton) {
      NewtonStats* nw = &a.host->nwt;
      host_store(&nw->r2, r2);
      host_store(&nw->fext2, f2);
      host_store(&nw->dU2, sm[0]);
      host_store(&nw->U2, sm[1]);
      if (a.tol.forcing) {  // every workgroup has passed its reading of the old one
        a.sc->nwt.prev_b2 = bb;
        host_store(&nw->prev_b2, bb);
        host_store(&nw->eta, eta);
      }
    }
  }
}

// Restarted GMRES(m) with right block-Jacobi preconditioning (K D^-1 y = b,
// x = D^-1 y), classical Gram-Schmidt twice, as gmres_solve_t in
// solver_kernels.hip, whose iteration is some ten launches and three host round
// trips: 157 us at 720 nodes in FP64, and 7.2 us here (289 -> 14.4 ms for the two
// load steps of a 9 x 8 x 7 box).  A workgroup holds R = T / L rows: the
// tangent in registers, the basis V of its 3 R dofs and the working vector w in
// LDS, the Hessenberg column in LDS and its rotations in the lanes of every wave.
// An iteration waits for the other workgroups three times: for the neighbours'
// t = D^-1 w (handed over as z of the PCG) and for the dot products of the two
// Gram-Schmidt passes (a value per basis vector, four threads a value).  |w| after
// the second pass comes with it: |w|^2 before it less the squares of its
// coefficients, all summed in FP64; where these take most of |w|^2 away it is
// summed again.  It lacks the rounding of the stored w, whose entries' errors average
// out: basis vectors of three boxes (a host model, 60 each) have a norm within 0.09 u of
// one in FP32 with either sum, and within 0.10 u instead of 0.08 u in FP64.  The rotations run while t is under way.  With |w| as an exchange
// of its own and slots polled one after the other an iteration was 14.5 us.
constexpr int kGmresThreads = 256;
constexpr int kGmresMax = 60;    // most basis vectors of the resident kernel (four threads each)
constexpr int kGmresSlot = 128;  // words of a workgroup's slot: 64 values

template <typename KT>
struct GmresArgs {
  const int32_t* sell_ptr;
  const int32_t* slice_rounds;
  int64_t rstride;
  const int32_t* scol;
  const KT* sval;
  const KT* Dinv;
  const double* b;
  const uint8_t* mask;
  KT* x;
  unsigned long long* t;  // D^-1 w, handed from workgroup to workgroup (share_node)
  PcgState* st;
  unsigned long long* slots;  // four regions of kMaxGridWg slots
  uint32_t base;
  int nwg, xcd;
  long long limit;
  int64_t nn;
  int m, maxiter;
  double rtol;
};

// LDS of one workgroup: packed triangle of R, two coefficient columns (the second
// with |w|^2), right-hand side, solution, two scalars; then w and the m + 1 basis
// vectors, each padded by 4 values so that four threads of 16 vectors hit distinct
// banks
inline size_t gmres_lds(int m, int rows, size_t kt) {
  return sizeof(double) * ((size_t)m * (m + 1) / 2 + 4 * 64 + 2) +
         kt * (size_t)(m + 2) * (3 * rows + 4);
}

template <typename KT, int L, int NB, Meet M>
__global__ __launch_bounds__(kGmresThreads) void k_gmres_resident(GmresArgs<KT> a) {
  constexpr int T = kGmresThreads, R = T / L, DN = 3 * R, S = DN + 4;
  constexpr int kSpread = M == Meet::kXcd ? 8 : 1;
  if (M == Meet::kXcd && (int)(blockIdx.x % kSpread) != a.xcd) return;
  const int wg = (int)(blockIdx.x / kSpread);
  extern __shared__ double lds[];
  __shared__ int late;  // a wait for t or x has expired
  const int m = a.m;
  double* Rm = lds;  // column j at j (j + 1) / 2
  double* h1 = Rm + m * (m + 1) / 2;
  double *h2 = h1 + 64, *gv = h2 + 64, *yv = gv + 64, *sc = yv + 64;
  KT* w = (KT*)(sc + 2);
  KT* V = w + S;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int ph = t % L, lrow = t / L;
  const int64_t i = (int64_t)wg * R + lrow;
  const bool row = i < a.nn;
  // a thread's dof (t < DN)
  const bool isd = t < DN;
  const int comp = t % 3, n0 = t - comp;
  const int64_t dof = (int64_t)wg * DN + t;
  const bool live = isd && dof < 3 * a.nn;
  const bool freed = live && !((a.mask[live ? dof / 3 : 0] >> comp) & 1u);
  const double bd = freed ? a.b[dof] : 0.0;
  // the node that this thread hands over (FP64: a half of it)
  const int gnode = t / kShareLanes<KT>, gpart = t % kShareLanes<KT>;
  const uint32_t gi = (uint32_t)(wg * R + gnode);
  const bool gives = gnode < R && gi < a.nn;
  KT gd[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) gd[q] = gives ? a.Dinv[9 * (int64_t)gi + q] : KT(0);
  KT d0 = 0, d1 = 0, d2 = 0, xs = 0;
  if (live) {
    const KT* D = a.Dinv + 9 * (dof / 3) + 3 * comp;
    d0 = D[0];
    d1 = D[1];
    d2 = D[2];
  }
  KT v[NB][9];
  uint32_t cj[NB];
  {
    const int64_t s = row ? i >> 6 : 0;
    const int32_t b0 = a.sell_ptr[s], rounds = a.slice_rounds[s];
    const int l = (int)(i & 63);
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int mr = ph + L * q;
      const bool has = row && mr < rounds;
      const int64_t b = b0 + a.rstride * (has ? mr : 0);
      cj[q] = has ? kShareBytes<KT> * (uint32_t)a.scol[b + l] : 0u;
#pragma unroll
      for (int e = 0; e < 9; ++e) v[q][e] = has ? a.sval[9 * b + 64 * e + l] : KT(0);
    }
  }
  if (t == 0) late = 0;
  __syncthreads();
  const GridSlots gs{a.slots, a.nwg, wg, &a.st->aborted, a.limit};
  const SharedBuf tbuf = shared_buf(a.t, kShareBytes<KT> * (uint32_t)a.nn);
  uint32_t ep = a.base;
  // w = scale K y, y the vector shared at this epoch
  auto product = [&](double scale) {
    KT yj[NB][3];
    if (!gather_shared<M, KT, NB>(tbuf, cj, ep, gs, yj)) late = 1;
    KT a0 = 0, a1 = 0, a2 = 0;
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      a0 += v[q][0] * yj[q][0] + v[q][1] * yj[q][1] + v[q][2] * yj[q][2];
      a1 += v[q][3] * yj[q][0] + v[q][4] * yj[q][1] + v[q][5] * yj[q][2];
      a2 += v[q][6] * yj[q][0] + v[q][7] * yj[q][1] + v[q][8] * yj[q][2];
    }
    a0 = group_sum<L>(a0);
    a1 = group_sum<L>(a1);
    a2 = group_sum<L>(a2);
    __syncthreads();  // the last readers of w are done
    if (ph < 3) {
      const KT ac = ph == 0 ? a0 : (ph == 1 ? a1 : a2);
      w[3 * lrow + ph] = (KT)((double)ac * scale);
    }
    __syncthreads();
  };
  // sum over the launch of `nval` values, four threads a value (acc: the thread's
  // part), to h
  auto share = [&](int nval, double acc, double* h, auto m) -> bool {
    constexpr Meet W = decltype(m)::value;
    ++ep;
    const int q = t >> 2, seg = t & 3;
    acc = group_sum<4>(acc);
    unsigned long long* reg =
        a.slots + (size_t)((ep & 1u) + (W == Meet::kXcd ? 2u : 0u)) * kMaxGridWg * kGmresSlot;
    bool ok = late == 0;
    double sum = 0;
    if (ok && q < nval) {
      if (seg < 2)
        shared_store<W>(reg + (size_t)kGmresSlot * wg + 2 * q + seg, value_word(acc, ep, seg));
      const SharedBuf rb = shared_buf(reg, 8u * kGmresSlot * kMaxGridWg);
      for (int g0 = seg; ok && g0 < gs.nwg; g0 += 16) {
        double x[4];
        uint32_t off[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          off[e] = 8u * (kGmresSlot * (g0 + 4 * e < gs.nwg ? g0 + 4 * e : wg) + 2 * q);
        ok = poll_values<W, 4>(rb, off, ep, gs, x);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          sum += g0 + 4 * e < gs.nwg ? x[e] : 0.0;
      }
    }
    sum = group_sum<4>(sum);
    if (q < nval && seg == 0) h[q] = sum;
    return __syncthreads_and(ok);
  };
  // h[0 .. nv) = V' w, and h[nv] = w' w with NORM
  auto dots = [&](int nv, double* h, bool norm) -> bool {
    const int q = t >> 2, seg = t & 3;
    const int nval = nv + (norm ? 1 : 0);
    double acc = 0, ac2 = 0;
    if (q < nval) {
      const KT* vq = q < nv ? V + q * S : w;
#pragma unroll 6
      for (int d = seg; d < DN; d += 8) {
        acc += (double)vq[d] * (double)w[d];
        ac2 += (double)vq[d + 4] * (double)w[d + 4];
      }
    }
    return share(nval, acc + ac2, h, std::integral_constant<Meet, M>());
  };
  auto subtract = [&](int nv, const double* h) {
    if (isd) {
      double s = 0;
#pragma unroll 4
      for (int q = 0; q < nv; ++q) s += h[q] * (double)V[q * S + t];
      w[t] = (KT)((double)w[t] - s);
    }
    __syncthreads();
  };
  // column j of the basis, w / |w|, and t = D^-1 w of the next product (K D^-1 v is
  // K t / |w|)
  auto next_column = [&](int j, double inv) {
    if (gives) {
      const KT x = w[3 * gnode], y = w[3 * gnode + 1], z = w[3 * gnode + 2];
      share_node<M>(tbuf, gi, gpart, gd[0] * x + gd[1] * y + gd[2] * z,
                 gd[3] * x + gd[4] * y + gd[5] * z, gd[6] * x + gd[7] * y + gd[8] * z, ep);
    }
    if (isd) V[j * S + t] = (KT)((double)w[t] * inv);
  };
  if (M == Meet::kXcd) {  // one XCD, as in k_pcg_resident: n sum x^2 = (sum x)^2
    const double x = t < 8 && (t & 3) == 0 ? (double)xcd_id() : 0.0;
    if (!share(2, t < 4 ? x : x * x, h1, std::integral_constant<Meet, Meet::kDevice>())) return;
    if (a.nwg * h1[1] != h1[0] * h1[0]) {
      if (t == 0) a.st->aborted = kNotOneXcd;
      return;
    }
    __syncthreads();
  }

  double beta0 = -1, beta = 0;
  int total = 0;
  for (bool first = true;; first = false) {
    // r = b - K x on the free dofs
    KT rv = freed ? (KT)bd : KT(0);
    if (!first) {
      // x at an epoch without a sum (two on, so that the sums' regions stay in turn);
      // the t that the last column left there is read by no one
      ep += 2;
      if (isd) w[t] = xs;
      __syncthreads();
      if (gives)
        share_node<M>(tbuf, gi, gpart, w[3 * gnode], w[3 * gnode + 1], w[3 * gnode + 2], ep);
      product(1.0);
      rv = freed ? (KT)(bd - (double)w[isd ? t : 0]) : KT(0);
      __syncthreads();
    }
    if (isd) w[t] = rv;
    __syncthreads();
    if (!dots(0, h1, true)) return;
    beta = sqrt(h1[0]);
    if (beta0 < 0) beta0 = beta;
    if (!(beta > a.rtol * beta0) || total >= a.maxiter || beta0 == 0) break;
    double inv = 1.0 / beta;
    next_column(0, inv);
    double g = beta, cs = 0, sn = 0;  // lane q of every wave: rotation q
    int k = 0;
    for (int j = 0; j < m; ++j) {
      product(inv);
      if (!dots(j + 1, h1, false)) return;
      subtract(j + 1, h1);
      if (!dots(j + 1, h2, true)) return;
      subtract(j + 1, h2);
      const double n1 = h2[j + 1], c2 = lane <= j ? h2[lane] : 0.0;
      double n2 = n1 - wave_sum(c2 * c2);
      if (n2 < 0.25 * n1) {  // the same answer in every workgroup
        if (!dots(0, h1 + 63, true)) return;
        n2 = h1[63];
      }
      const double hn = sqrt(n2);
      if (hn > 0) {
        inv = 1.0 / hn;
        next_column(j + 1, inv);
      }
      // the earlier rotations applied to the new column
      const double col = lane <= j ? h1[lane] + h2[lane] : 0.0;
      double e = read_lane(col, 0), mine = 0;
      for (int q = 0; q < j; ++q) {
        const double f = read_lane(col, q + 1), cq = read_lane(cs, q), sq = read_lane(sn, q);
        if (lane == q) mine = cq * e + sq * f;
        e = cq * f - sq * e;
      }
      const double r = hypot(e, hn);
      const double c = r > 0 ? e / r : 1.0, s = r > 0 ? hn / r : 0.0;
      if (lane == j) {
        cs = c;
        sn = s;
        mine = r;
      }
      if (t <= j) Rm[j * (j + 1) / 2 + t] = mine;
      if (t == j) gv[j] = c * g;
      g = -s * g;
      ++total;
      k = j + 1;
      if (fabs(g) <= a.rtol * beta0 || total >= a.maxiter || !(hn > 0)) break;
    }
    __syncthreads();
    if (t < 64) {  // R y = g, a lane per unknown
      double y = lane < k ? gv[lane] : 0.0;
      for (int q = k - 1; q >= 0; --q) {
        const double* col = Rm + q * (q + 1) / 2;
        const double d = col[q];
        const double yq = d != 0 ? read_lane(y, q) / d : 0.0;
        if (lane < q) y -= col[lane] * yq;
        if (lane == q) yv[q] = yq;
      }
    }
    __syncthreads();
    if (isd) {
      double s = 0;
      for (int q = 0; q < k; ++q) s += yv[q] * (double)V[q * S + t];
      w[t] = (KT)s;
    }
    __syncthreads();
    if (live) xs += d0 * w[n0] + d1 * w[n0 + 1] + d2 * w[n0 + 2];
    __syncthreads();
  }
  if (live) a.x[dof] = xs;
  if (wg == 0 && t == 0) {
    a.st->rr_last = beta * beta;
    a.st->bb = beta0 * beta0;
    a.st->iters = total;
    a.st->k = (int32_t)(ep - a.base);  // epochs used
    a.st->converged = (beta0 == 0 || beta <= a.rtol * beta0) ? 1 : 0;
    a.st->done = 1;
  }
}

// L lanes a row: 4 for rows of up to 16 blocks (structured meshes: 15), 8 up to 32
inline int lanes_per_row(const Ctx* c) { return c->ell_width <= 16 ? 4 : 8; }
constexpr int kResidentBlocks = 4;  // blocks a lane keeps in registers
// Threads a workgroup: few, because an exchange waits for the workgroup's own barriers
// too.  Newton solves of 1,680 / 4,096 nodes took 14.9 / - ms with 128 threads, 14.8 /
// 9.7 ms with 256 and 15.5 / 10.2 ms with 512 across the device, against 49.6 ms on two
// kernels an iteration; of 4,913 / 6,859 / 8,000 nodes 9.4 / 12.9 / 13.7 ms with 256 (the
// first in one XCD) and 13.6 / 13.8 / 15.7 ms with 512, which are left for more than
// kMaxGridWg workgroups of 256.  The single workgroup gathers from LDS: 512 threads, and
// in FP32 1024 where the rows need them (125 nodes: 1.0 us an iteration against 2.0 on
// several workgroups, 252 nodes: 1.7 against 2.2; FP64, 125 nodes: 1.2 against 2.5).
constexpr int kResidentThreads = 256;
constexpr int resident_one_threads(size_t kt) { return kt == 4 ? 1024 : 512; }

// where a launch's workgroups meet (an index of Ctx::resident_launches)
enum Place { kOneWorkgroup, kOneXcd, kAcrossDevice, kGaveUp };

struct ResidentShape {
  int threads;
  int64_t grid;
};
inline ResidentShape resident_shape(const Ctx* c) {
  const int64_t lanes = c->nn * lanes_per_row(c);
  if (lanes <= 512) return {512, 1};
  if (lanes <= resident_one_threads(c->kt)) return {resident_one_threads(c->kt), 1};
  int t = kResidentThreads;
  if ((lanes + t - 1) / t > kMaxGridWg) t *= 2;
  return {t, (lanes + t - 1) / t};
}

// Every 8th workgroup of a launch shares an XCD: 32 CUs, on which 64 workgroups of 256
// threads are resident together with two waves a SIMD (FP64), and 96 with three (FP32).
// That many do better there, met in its L2, than spread over the device: FP32 1,680 /
// 4,096 / 5,832 nodes 10.3 / 7.6 / 9.8 ms against 14.1 / 9.6 / 12.6 ms, FP64 2,080 /
// 3,375 nodes 2.8 / 9.4 ms against 3.8 / 11.2 ms, GMRES at 720 nodes 14.4 ms against
// 17.3 ms.
inline bool on_one_xcd(const Ctx* c, int64_t grid, int blocks) {
  return c->one_xcd && fits_one_xcd(grid, blocks, c->cus);
}

// workgroups of `kern` that a CU takes
template <typename... A>
int blocks_per_cu(Ctx* c, void (*kern)(A...), int threads, size_t lds, int* blocks) {
  ONSAS_HIP_TRY(c, hipOccupancyMaxActiveBlocksPerMultiprocessor(
                       blocks, reinterpret_cast<const void*>(kern), threads, lds));
  return ONSAS_OK;
}
inline size_t share_words(const Ctx* c) { return (size_t)c->nn * c->kt / 2; }  // kShareBytes a node

// f(kernel of a shape, its threads, its grid)
template <typename KT, int L, typename F>
int with_pcg_kernel(const ResidentShape& sh, bool xcd, F f) {
  constexpr int T1 = resident_one_threads(sizeof(KT)), T = kResidentThreads;
  constexpr int NB = kResidentBlocks;
  constexpr Meet D = Meet::kDevice, X = Meet::kXcd;
  if (sh.grid == 1 && sh.threads == 512) return f(k_pcg_resident<KT, L, NB, 512, true, D>, 512, 1);
  if (sh.grid == 1) return f(k_pcg_resident<KT, L, NB, T1, true, D>, T1, 1);
  if (xcd) return f(k_pcg_resident<KT, L, NB, T, false, X>, T, 8 * sh.grid);
  if (sh.threads == T) return f(k_pcg_resident<KT, L, NB, T, false, D>, T, sh.grid);
  return f(k_pcg_resident<KT, L, NB, 2 * T, false, D>, 2 * T, sh.grid);
}

// Where the model's PCG may meet, from what the device takes of its kernels.
template <typename KT, int L>
int pcg_places(Ctx* c) {
  const ResidentShape sh = resident_shape(c);
  auto blocks = [&](bool xcd, int* n) -> int {
    return with_pcg_kernel<KT, L>(sh, xcd, [&](auto kern, int threads, int64_t) {
      return blocks_per_cu(c, kern, threads, 0, n);
    });
  };
  int n = 0;
  ONSAS_TRY(blocks(false, &n));
  c->pcg_device = fits_device(sh.grid, n, c->cus);
  c->pcg_xcd = false;
  if (sh.grid > 1 && sh.threads == kResidentThreads) {
    ONSAS_TRY(blocks(true, &n));
    c->pcg_xcd = fits_one_xcd(sh.grid, n, c->cus);
  }
  return ONSAS_OK;
}

// the longest wait of the next launch
inline long long wait_ticks(Ctx* c) {
  if (c->first_launches == 0) return c->gslot_ticks;
  --c->first_launches;
  return c->first_ticks;
}

// A Newton step's launch stamps the step's timing events.
template <typename KT, int L>
int run_resident(Ctx* c, const ResidentArgs<KT>& a, const ResidentShape& sh, bool xcd) {
  const hipEvent_t e0 = a.fint ? c->ev[4] : nullptr, e1 = a.fint ? c->ev[7] : nullptr;
  return with_pcg_kernel<KT, L>(sh, xcd, [&](auto kern, int threads, int64_t grid) -> int {
    hipExtLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(threads), 0, c->stream, e0, e1, 0, a);
    ONSAS_HIP_TRY(c, hipGetLastError());
    return ONSAS_OK;
  });
}

template <typename KT>
int resident_t(Ctx* c, const double* b, const double* fint, const void* x0, void* warm, Place* at) {
  ResidentArgs<KT> a{};
  a.sell_ptr = c->d_sell_ptr;
  a.slice_rounds = c->d_slice_rounds;
  a.rstride = c->ell_rounds ? 64 * c->nslices : 64;
  a.scol = c->d_sell_col;
  a.sval = (const KT*)c->d_Ksell;
  a.Dinv = (const KT*)c->d_Dinv;
  a.mask = c->d_fixmask;
  a.b = b;
  a.x = (KT*)c->d_px;
  a.z = c->d_share;
  a.sc = c->d_sc;
  a.host = c->h_sc;
  a.slots = c->d_gslots;
  a.maxiter = pcg_maxiter(c);
  a.tol = inner_tol(c, fint != nullptr);
  a.fint = fint;
  a.x0 = (const KT*)x0;
  a.warm = (KT*)warm;
  a.res = c->d_res;
  a.U = c->d_U;
  a.base = c->gslot_epoch;
  a.limit = wait_ticks(c);
  a.nn = c->nn;
  const ResidentShape sh = resident_shape(c);
  const bool xcd = c->one_xcd && c->pcg_xcd;
  *at = sh.grid == 1 ? kOneWorkgroup : xcd ? kOneXcd : kAcrossDevice;
  a.nwg = (int)sh.grid;
  a.xcd = c->xcd;
  return lanes_per_row(c) == 4 ? run_resident<KT, 4>(c, a, sh, xcd)
                               : run_resident<KT, 8>(c, a, sh, xcd);
}

template <typename KT, int L>
int gmres_t(Ctx* c, const double* b_dev, int m, int maxiter, double rtol, Place* at) {
  GmresArgs<KT> a{};
  a.sell_ptr = c->d_sell_ptr;
  a.slice_rounds = c->d_slice_rounds;
  a.rstride = c->ell_rounds ? 64 * c->nslices : 64;
  a.scol = c->d_sell_col;
  a.sval = (const KT*)c->d_Ksell;
  a.Dinv = (const KT*)c->d_Dinv;
  a.b = b_dev;
  a.mask = c->d_fixmask;
  a.x = (KT*)c->d_px;
  a.t = c->d_share;
  a.st = &c->d_sc->pcg;
  a.slots = c->d_gmslots;
  a.base = c->gslot_epoch;
  a.limit = wait_ticks(c);
  a.nn = c->nn;
  a.m = m;
  a.maxiter = maxiter;
  a.rtol = rtol;
  const int R = kGmresThreads / L;
  const int64_t grid = (c->nn + R - 1) / R;
  a.nwg = (int)grid;
  a.xcd = c->xcd;
  const size_t lds = gmres_lds(m, R, sizeof(KT));
  // *at = kGaveUp: the device does not take the grid, and nothing has been launched
  auto blocks = [&](auto kern, int* n) -> int {
    ONSAS_HIP_TRY(c, hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    return blocks_per_cu(c, kern, kGmresThreads, lds, n);
  };
  auto go = [&](auto kern, int64_t n) -> int {
    hipLaunchKernelGGL(kern, dim3((unsigned)n), dim3(kGmresThreads), lds, c->stream, a);
    ONSAS_HIP_TRY(c, hipGetLastError());
    return ONSAS_OK;
  };
  int n = 0;
  ONSAS_TRY(blocks(k_gmres_resident<KT, L, kResidentBlocks, Meet::kXcd>, &n));
  if (on_one_xcd(c, grid, n)) {
    *at = kOneXcd;
    return go(k_gmres_resident<KT, L, kResidentBlocks, Meet::kXcd>, 8 * grid);
  }
  ONSAS_TRY(blocks(k_gmres_resident<KT, L, kResidentBlocks, Meet::kDevice>, &n));
  *at = fits_device(grid, n, c->cus) ? kAcrossDevice : kGaveUp;
  return *at == kGaveUp ? ONSAS_OK : go(k_gmres_resident<KT, L, kResidentBlocks, Meet::kDevice>, grid);
}

}  // namespace

// Solves that a context takes on the slower path before it tries again, doubled by every
// launch that gives up and back to the first by one that solves: an expired wait is 0.2 s,
// some tens of general solves, so a GPU that stays busy costs a vanishing share of it and
// one that was busy once costs a model this many slower solves.
constexpr int kFirstRest = 64, kLongestRest = 1 << 16;

// Whether a block-Jacobi PCG of this model runs as one launch: rows short enough
// for the lanes' registers and a grid of at most kMaxGridWg workgroups (16,384
// rows of up to 16 blocks, 8,192 of up to 32).
bool pcg_resident_fits(const Ctx* c) {
  return kSellLanes == 1 && c->ell_width <= 8 * kResidentBlocks &&
         resident_shape(c).grid <= kMaxGridWg;
}

int pcg_resident_setup(Ctx* c) {
  const char* e = std::getenv("ONSAS_PCG_RESIDENT");
  c->pcg_resident = c->may_pcg_resident = pcg_resident_fits(c) && !(e && e[0] == '0');
  if (const char* x = std::getenv("ONSAS_RESIDENT_XCD")) c->one_xcd = c->may_one_xcd = x[0] != '0';
  c->resident_rest = 0;
  c->resident_pause = kFirstRest;
  // "n" ticks, or "n:m", for the first m launches
  if (const char* t = std::getenv("ONSAS_RESIDENT_TICKS")) {
    const char* colon = std::strchr(t, ':');
    (colon ? c->first_ticks : c->gslot_ticks) = std::atoll(t);
    c->first_launches = colon ? std::atoi(colon + 1) : 0;
  }
  static std::atomic<unsigned> contexts{0};
  c->xcd = (int)((contexts++ + (unsigned)getpid()) % 8);
  if (!c->pcg_resident) return ONSAS_OK;
  ONSAS_HIP_TRY(c, hipDeviceGetAttribute(&c->cus, hipDeviceAttributeMultiprocessorCount, c->device));
  const bool f64 = c->precision == ONSAS_PRECISION_FP64;
  if (lanes_per_row(c) == 4)
    ONSAS_TRY(f64 ? (pcg_places<double, 4>(c)) : (pcg_places<float, 4>(c)));
  else
    ONSAS_TRY(f64 ? (pcg_places<double, 8>(c)) : (pcg_places<float, 8>(c)));
  const size_t bytes = share_words(c) * sizeof(unsigned long long);
  ONSAS_HIP_TRY(c, hipMalloc((void**)&c->d_share, bytes));
  ONSAS_HIP_TRY(c, hipMemset(c->d_share, 0, bytes));
  return ONSAS_OK;
}

// the abort word of a launch that gave up
static int clear_abort(Ctx* c) {
  ONSAS_HIP_TRY(c, hipMemsetAsync(&c->d_sc->pcg.aborted, 0, sizeof(int32_t), c->stream));
  return ONSAS_OK;
}

// before the epochs wrap: clear the marks and begin again
static int renew_epochs(Ctx* c) {
  if (c->gslot_epoch <= 0xf0000000u) return ONSAS_OK;
  ONSAS_HIP_TRY(c, hipMemsetAsync(c->d_gslots, 0,
                                  kGridSlotWords * sizeof(unsigned long long), c->stream));
  ONSAS_HIP_TRY(c, hipMemsetAsync(c->d_share, 0, share_words(c) * sizeof(unsigned long long),
                                  c->stream));
  if (c->d_gmslots)
    ONSAS_HIP_TRY(c, hipMemsetAsync(c->d_gmslots, 0, 4 * (size_t)kMaxGridWg * kGmresSlot *
                                                         sizeof(unsigned long long), c->stream));
  c->gslot_epoch = 1;
  return ONSAS_OK;
}

// A launch that gave up (a wait expired: the GPU, or the XCD, was too busy to hold the
// whole grid) or found its workgroups on several XCDs: the next one meets across the
// device, and after that the context keeps to the general kernels, for some solves.
static void resident_failed(Ctx* c, Place at) {
  c->resident_launches[kGaveUp]++;
  if (at == kOneXcd)
    c->one_xcd = false;
  else
    c->pcg_resident = false;
  c->resident_rest = c->resident_pause;
  c->resident_pause = std::min(2 * c->resident_pause, kLongestRest);
}
static void resident_solved(Ctx* c, Place at) {
  c->resident_launches[at]++;
  if (c->resident_rest == 0) c->resident_pause = kFirstRest;
}
// before a solve that may be one launch: back to the fastest path once the rest is over
static void resident_turn(Ctx* c) {
  if (c->resident_rest == 0 || --c->resident_rest > 0) return;
  c->one_xcd = c->may_one_xcd;
  c->pcg_resident = c->may_pcg_resident;
}

// Launches, waits and takes the results; *ran = false if the launch gave up.
static int resident_run(Ctx* c, const double* b, const double* fint, const void* x0, void* warm,
                        bool* ran, int* iters, double* relres, int* converged, int* breakdown) {
  ONSAS_TRY(renew_epochs(c));
  c->h_sc->pcg = PcgState{};
  Place at = kOneWorkgroup;
  ONSAS_TRY(c->precision == ONSAS_PRECISION_FP64 ? resident_t<double>(c, b, fint, x0, warm, &at)
                                                 : resident_t<float>(c, b, fint, x0, warm, &at));
  ONSAS_HIP_TRY(c, hipStreamSynchronize(c->stream));
  const PcgState& ps = c->h_sc->pcg;
  *ran = ps.done && !ps.aborted;
  // an iteration takes at most two epochs
  c->gslot_epoch += (*ran ? (uint32_t)ps.k : 2 * (uint32_t)pcg_maxiter(c) + 5) + 1;
  if (*ran) {
    resident_solved(c, at);
    pcg_result(ps, iters, relres, converged, breakdown);
    return ONSAS_OK;
  }
  resident_failed(c, at);
  return clear_abort(c);
}

inline bool pcg_resident_kind(const Ctx* c) {
  return c->may_pcg_resident && c->lin.precond != ONSAS_PRECOND_AMG &&
         pcg_maxiter(c) <= kMaxResidentIters;
}
inline bool pcg_resident_now(const Ctx* c) {
  return c->pcg_resident && (c->pcg_device || (c->one_xcd && c->pcg_xcd));
}

int launch_pcg_resident(Ctx* c, const double* b_dev, bool* ran, int* iters, double* relres,
                        int* converged, int* breakdown) {
  *ran = false;
  if (!pcg_resident_kind(c)) return ONSAS_OK;
  resident_turn(c);
  while (!*ran && pcg_resident_now(c))
    ONSAS_TRY(resident_run(c, b_dev, nullptr, nullptr, nullptr, ran, iters, relres, converged,
                           breakdown));
  return ONSAS_OK;
}

int launch_newton_resident(Ctx* c, const void* x0, void* warm, bool* ran, int* iters,
                           double* relres, int* converged, int* breakdown) {
  *ran = false;
  if (!pcg_resident_kind(c) || c->lin.kind == ONSAS_LINSOLVE_GMRES) return ONSAS_OK;
  resident_turn(c);
  while (!*ran && pcg_resident_now(c)) {
    const double prev_b2 = c->h_sc->nwt.prev_b2;
    ONSAS_TRY(resident_run(c, c->d_fext, c->d_fint, x0, warm, ran, iters, relres, converged,
                           breakdown));
    if (*ran) break;
    // U and the forcing's memory as they were (some workgroups may have got that far)
    ONSAS_HIP_TRY(c, hipMemcpyAsync(c->d_U, c->d_Uasm, 3 * c->nn * sizeof(double),
                                    hipMemcpyDeviceToDevice, c->stream));
    c->h_sc->nwt.prev_b2 = prev_b2;
    ONSAS_HIP_TRY(c, hipMemcpyAsync(&c->d_sc->nwt.prev_b2, &c->h_sc->nwt.prev_b2, sizeof(double),
                                    hipMemcpyHostToDevice, c->stream));
  }
  return ONSAS_OK;
}

// GMRES of the current tangent in one launch, where the model and the restart
// length fit (a basis of up to kGmresMax vectors in 150 KiB of LDS a workgroup);
// *ran = false leaves the solve to the general path.
int launch_gmres_resident(Ctx* c, const double* b_dev, int m, int maxiter, double rtol, bool* ran,
                          int* iters, double* relres, int* converged) {
  *ran = false;
  const int L = lanes_per_row(c), R = kGmresThreads / L;
  if (!c->may_pcg_resident || m > kGmresMax || maxiter > kMaxResidentIters ||
      (c->nn + R - 1) / R > kMaxGridWg || gmres_lds(m, R, c->kt) > 150 * 1024)
    return ONSAS_OK;
  hipStream_t s = c->stream;
  const size_t bytes = 4 * (size_t)kMaxGridWg * kGmresSlot * sizeof(unsigned long long);
  resident_turn(c);
  while (!*ran && c->pcg_resident) {
    if (!c->d_gmslots) {
      ONSAS_HIP_TRY(c, hipMalloc((void**)&c->d_gmslots, bytes));
      ONSAS_HIP_TRY(c, hipMemsetAsync(c->d_gmslots, 0, bytes, s));
    }
    ONSAS_TRY(renew_epochs(c));
    ONSAS_HIP_TRY(c, hipMemsetAsync(&c->d_sc->pcg, 0, sizeof(PcgState), s));
    Place at = kOneXcd;
    if (c->precision == ONSAS_PRECISION_FP64)
      ONSAS_TRY(L == 4 ? (gmres_t<double, 4>(c, b_dev, m, maxiter, rtol, &at))
                       : (gmres_t<double, 8>(c, b_dev, m, maxiter, rtol, &at)));
    else
      ONSAS_TRY(L == 4 ? (gmres_t<float, 4>(c, b_dev, m, maxiter, rtol, &at))
                       : (gmres_t<float, 8>(c, b_dev, m, maxiter, rtol, &at)));
    if (at == kGaveUp) return ONSAS_OK;
    ONSAS_HIP_TRY(c, hipMemcpyAsync(&c->h_sc->pcg, &c->d_sc->pcg, sizeof(PcgState),
                                    hipMemcpyDeviceToHost, s));
    ONSAS_HIP_TRY(c, hipStreamSynchronize(s));
    const PcgState& ps = c->h_sc->pcg;
    *ran = !ps.aborted;
    // an iteration takes at most 3 epochs, a restart 3
    c->gslot_epoch += (*ran ? (uint32_t)ps.k : 6u * ((uint32_t)maxiter + 2)) + 4;
    if (*ran) {
      resident_solved(c, at);
      *iters = ps.iters;
      *relres = ps.bb > 0 ? std::sqrt(ps.rr_last / ps.bb) : 0.0;
      *converged = ps.converged;
    } else {
      resident_failed(c, at);
      ONSAS_TRY(clear_abort(c));
    }
  }
  return ONSAS_OK;
}

}  // namespace onsas
