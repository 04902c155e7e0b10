// inner_tol.hpp -- stopping tolerance of the inner (linear) solve, applied by the
// kernels that start one.
#pragma once

#include <hip/hip_runtime.h>

namespace onsas {

// Fixed: ||r|| <= rtol ||b||.  Forcing (inexact Newton): eta = max(0.9 (||b_k|| /
// ||b_{k-1}||)^2 [Eisenstat-Walker choice 2, gamma = 0.9, alpha = 2],
// kForcingGuard tau / ||b_k||) clamped to [rtol, eta_max], where b_k is this
// Newton iteration's residual and tau = newton_tol ||f_ext|| the outer target: no
// inner accuracy is bought beyond what the quadratic model or the outer tolerance
// can use.  The first iteration of a load step uses eta_first.
//
// kForcingGuard = 0.5 is the safeguard of C. T. Kelley, Iterative Methods for
// Linear and Nonlinear Equations (SIAM 1995), sec. 6.3.  On the 64^3 cube
// (80 Newton iterations at every factor tried) it took the mixed solve from
// 425 PCG iterations / 0.149 s at 0.1 to 379 / 0.137 s (FP64 384 -> 350),
// with 1.0 at 363 / 0.133 s: 0.5 keeps the last inner solve a factor of two
// inside the outer tolerance.
constexpr double kForcingGuard = 0.5;

struct InnerTol {
  double rtol, newton_tol, eta_max, eta_first;
  int forcing;
};

// bb = ||b_k||^2, ff = ||f_ext||^2 and prev = ||b_{k-1}||^2 (0: none), the latter
// two with forcing only
__device__ inline double inner_eta(const InnerTol& t, double bb, double ff, double prev) {
  if (!t.forcing) return t.rtol;
  const double tau = t.newton_tol * sqrt(ff);
  double e = prev > 0 ? 0.9 * (bb / prev) : t.eta_first;
  if (bb > 0) e = fmax(e, kForcingGuard * tau / sqrt(bb));
  // the residual already meets the outer tolerance: this solve only refines
  // (the reference applies it before its convergence test sees the residual)
  const double cap = (bb > 0 && sqrt(bb) <= tau) ? fmax(t.eta_max, 0.5) : t.eta_max;
  return fmin(fmax(e, t.rtol), cap);
}

}  // namespace onsas
