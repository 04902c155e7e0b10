"""The multigrid-preconditioned CG against the same iteration in numpy, on the
hierarchy copied back from the device: the V-cycle's products, transfers and
coarse solve all enter the iteration count and the iterates."""
import numpy as np
import pytest

from onsas_amd import _capi, meshes
from onsas_amd._capi import Context

pytestmark = pytest.mark.gpu


def _model(prec, nx, ny, nz):
    sm = meshes.cube(nx, ny=ny, nz=nz, jitter=0.05, seed=4)
    c = Context(prec)
    c.set_nodes(sm.coords)
    c.add_tet_group(sm.tets, _capi.MAT_NEOHOOKEAN, (8.3e5, 3.8e5))
    c.set_fixed_dofs((3 * sm.node_sets["x0"][:, None] + np.arange(3)).reshape(-1))
    c.finalize()
    return c, sm.nn


def _block_inverses(A, bs):
    n = A.shape[0] // bs
    D = np.zeros((n, bs, bs))
    A = A.tobsr((bs, bs))
    rows = np.repeat(np.arange(n), np.diff(A.indptr))
    D[rows[rows == A.indices]] = A.data[rows == A.indices]
    return np.linalg.inv(D)


class Cycle:
    """The V-cycle of amg.hip's header comment in FP64."""

    def __init__(self, c):
        self.lev = []
        nl = c.amg_levels()
        for l in range(nl):
            info = c.amg_level_info(l)
            A = c.tangent_bsr() if l == 0 else c.amg_operator(l)
            if l + 1 == nl:  # solved exactly
                self.lev.append(dict(A=A.tocsr(), P=None))
                break
            hi = 1.1 * info["lam"]
            lo = hi / 30
            th, de = (hi + lo) / 2, (hi - lo) / 2
            rho0 = de / th
            rho1 = 1 / (2 / rho0 - rho0)
            self.lev.append(dict(A=A.tocsr(), th=th, c1=rho1 * rho0, c2=2 * rho1 / de, bs=info["bs"],
                                 P=c.amg_prolongator(l).tocsr(), D=_block_inverses(A, info["bs"])))

    def __call__(self, b, l=0):
        L = self.lev[l]
        A = L["A"]
        if L["P"] is None:
            A = A.toarray()
            A[A.diagonal() == 0, A.diagonal() == 0] = 1.0  # a vanished coarse dof: unit diagonal
            return np.linalg.solve(A, b)
        Dinv = lambda r: np.einsum("nij,nj->ni", L["D"], r.reshape(-1, L["bs"])).reshape(-1)

        def smooth(r):
            d0 = Dinv(r) / L["th"]
            return d0 if l == 0 else d0 + L["c1"] * d0 + L["c2"] * Dinv(r - A @ d0)
        x = smooth(b)
        x = x + L["P"] @ self(L["P"].T @ (b - A @ x), l + 1)
        return x + smooth(b - A @ x)


def _pcg(A, M, b, rtol):
    x, r = np.zeros_like(b), b.copy()
    z = M(r)
    p, rz, k = z, r @ z, 0
    while np.linalg.norm(r) > rtol * np.linalg.norm(b) and k < 200:
        q = A @ p
        a = rz / (p @ q)
        x, r = x + a * p, r - a * q
        z = M(r)
        rz, old = r @ z, rz
        p, k = z + rz / old * p, k + 1
    return x, k


# nodes: 8 (one aggregate), 60, 480 and 1,430 (two levels), 9,261 (three, a coarse
# level of wave-per-row products), 57,967 (a coarse level in sliced ELL)
@pytest.mark.parametrize("prec", [_capi.PRECISION_MIXED, _capi.PRECISION_FP64])
@pytest.mark.parametrize("shape", [(1, 1, 1), (4, 3, 2), (9, 7, 5), (12, 10, 9), (20, 20, 20),
                                   (38, 37, 38)])
def test_cycle_matches_numpy(shape, prec):
    print(f"[gpu] cycle {shape} precision {prec}", flush=True)
    c, nn = _model(prec, *shape)
    try:
        rtol = 1e-4 if prec == _capi.PRECISION_MIXED else 1e-10
        c.set_linear_solver(_capi.LINSOLVE_PCG, rtol=rtol, precond=_capi.PRECOND_AMG)
        c.set_U(np.zeros(3 * nn))
        c.assemble()
        b = np.random.default_rng(nn).normal(size=3 * nn)
        x, it, _ = c.linear_solve(b)
        M = Cycle(c)
        A = M.lev[0]["A"]
        bf = np.where(x == 0, 0.0, b)
        xn, itn = _pcg(A, M, bf, rtol)
        # mixed mode rounds the cycle's vectors to FP32 and a large coarse level to
        # BF16 (2^-9, against a contraction of about 0.3 an iteration): the counts
        # may part by one; both iterates are within rtol of the solution
        assert abs(it - itn) <= 1, (it, itn)
        assert np.linalg.norm(bf - A @ x) <= 1.5 * rtol * np.linalg.norm(bf)
        if prec == _capi.PRECISION_FP64 and it == itn:
            # iterates of equal index agree to rounding, not only to rtol
            assert np.linalg.norm(x - xn) <= 1e-9 * np.linalg.norm(xn)
    finally:
        c.close()
