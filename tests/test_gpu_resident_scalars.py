"""The scalars of the one-launch PCG on tangents whose rounding shows: chains of 20 bars'
nodes with stiffnesses spread over seven decades, in FP32.

The general path sums p.q from p and q.  The launch makes it from sums that it takes
anyway and has to stay as good: where its rounding adds up over the iterations, search
directions lose their step lengths and the solves take more of them.  A host model of
both (the same recurrences in numpy, FP32 vectors and FP64 sums, 192 chains, three sets
of them and three orders of a row's additions) takes 24,037 to 25,208 iterations in
total with the direct sum, 24,120 to 25,637 with a p.q that starts from the stored
vectors each time, and 28,580 to 47,898, with solves that do not end, where it is
carried on."""
import numpy as np
import pytest

from onsas_amd import _capi
from onsas_amd._capi import Context

pytestmark = pytest.mark.gpu

CHAINS, NODES, DECADES = 192, 20, 7


def _definite(k):
    """The tangent stays positive definite when its entries are rounded to FP32, which moves
    the eigenvalues of the one scaled to a unit diagonal by at most 2 u."""
    K = np.diag(k[:-1] + k[1:]) - np.diag(k[1:-1], 1) - np.diag(k[1:-1], -1)
    d = 1 / np.sqrt(np.diag(K))
    return np.linalg.eigvalsh(d[:, None] * K * d)[0] > 2 * 2.0 ** -24


def _chains():
    for seed in range(3):
        r = np.random.default_rng(seed)
        k = 10 ** r.uniform(-DECADES / 2, DECADES / 2, (CHAINS // 3, NODES + 1))
        b = r.normal(size=(CHAINS // 3, NODES))
        yield from (kb for kb in zip(k, b) if _definite(kb[0]))


def _iterations(k, b, stride):
    """Iterations of one chain's solve; its nodes are `stride` apart in the numbering, the
    nodes between them belong to no element and are fixed."""
    at = stride * np.arange(NODES + 2)
    n = int(at[-1]) + 1
    X = np.stack([np.arange(n) / stride, np.zeros(n), np.zeros(n)], axis=1)
    c = Context(_capi.PRECISION_MIXED)
    try:
        c.set_nodes(X)
        c.add_truss_group(np.stack([at[:-1], at[1:]], axis=1), _capi.STRAIN_GREEN, 1.0, k)
        free = 3 * at[1:-1]
        c.set_fixed_dofs(np.setdiff1d(np.arange(3 * n), free))
        c.finalize()
        c.set_linear_solver(_capi.LINSOLVE_PCG, rtol=1e-6, maxiter=20000)
        c.set_U(np.zeros(3 * n))
        c.assemble()
        f = np.zeros(3 * n)
        f[free] = b
        return c.linear_solve(f)[1]
    finally:
        c.close()


@pytest.mark.parametrize("stride", [1, 25])  # 22 nodes: one workgroup; 526: nine
def test_step_lengths_of_stiffness_contrasts(monkeypatch, stride):
    print(f"[gpu] resident pcg, chains of bars, node stride {stride}", flush=True)
    it = sum(_iterations(k, b, stride) for k, b in _chains())
    monkeypatch.setenv("ONSAS_PCG_RESIDENT", "0")
    itg = sum(_iterations(k, b, stride) for k, b in _chains())
    print(f"iterations {it}, general path {itg}", flush=True)
    assert it <= 1.1 * itg
