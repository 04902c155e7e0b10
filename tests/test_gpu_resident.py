"""The one-launch block-Jacobi PCG and GMRES of small models (resident_solve.hip) at the
edges of its shapes: one workgroup and several, full and partial ones, 4 and 8
lanes a row, models just past its limits, and the path a launch takes when a
wait for the other workgroups expires."""
import numpy as np
import pytest

from onsas_amd import _capi, meshes
from onsas_amd._capi import Context

pytestmark = pytest.mark.gpu


def _box(prec, nx, ny, nz):
    sm = meshes.cube(nx, ny=ny, nz=nz, jitter=0.05, seed=4)
    c = Context(prec)
    c.set_nodes(sm.coords)
    c.add_tet_group(sm.tets, _capi.MAT_NEOHOOKEAN, (8.3e5, 3.8e5))
    c.set_fixed_dofs((3 * sm.node_sets["x0"][:, None] + np.arange(3)).reshape(-1))
    c.finalize()
    return c, sm.nn


def _clique(prec, n):
    """Bars between all pairs of n random nodes: every row has n blocks."""
    r = np.random.default_rng(n)
    X = r.uniform(0, 1, (n, 3))
    c = Context(prec)
    c.set_nodes(X)
    i, j = np.triu_indices(n, 1)
    c.add_truss_group(np.stack([i, j], axis=1), _capi.STRAIN_GREEN, 2e5, 1e-3)
    c.set_fixed_dofs(np.arange(9))
    c.finalize()
    return c, n


MODELS = {  # nodes: 8, 60, 128 / 140 (FP64 single workgroup ends at 128), 252 / 264 (FP32 at 256),
    # 1331 (several workgroups, the last one partial), 4352 (workgroups of twice the threads),
    # 9240 (more workgroups than one poll covers)
    "1x1x1": lambda p: _box(p, 1, 1, 1), "4x3x2": lambda p: _box(p, 4, 3, 2),
    "7x3x3": lambda p: _box(p, 7, 3, 3), "6x4x3": lambda p: _box(p, 6, 4, 3),
    "8x6x3": lambda p: _box(p, 8, 6, 3), "10x5x3": lambda p: _box(p, 10, 5, 3),
    "10x10x10": lambda p: _box(p, 10, 10, 10),
    "16x15x15": lambda p: _box(p, 16, 15, 15),
    "21x20x19": lambda p: _box(p, 21, 20, 19),
    "clique 17": lambda p: _clique(p, 17), "clique 32": lambda p: _clique(p, 32),
    "clique 33": lambda p: _clique(p, 33),  # rows too long: the general path
}


def _solve(make, prec, rtol, kind=_capi.LINSOLVE_PCG, restart=40):
    c, nn = make(prec)
    try:
        c.set_linear_solver(kind, rtol=rtol, gmres_restart=restart, maxiter=20000)
        c.set_U(np.zeros(3 * nn))
        c.assemble()
        K = c.tangent_bsr().tocsr()
        b = np.random.default_rng(nn).normal(size=3 * nn)
        x, it, _ = c.linear_solve(b)
        x2, it2, _ = c.linear_solve(b)
        assert it == it2 and np.array_equal(x, x2)  # deterministic, and the slots are reusable
        fixed = x == 0
        nb = np.linalg.norm(np.where(fixed, 0, b))
        res = np.linalg.norm(np.where(fixed, 0, b - K @ x)) / nb
        # the recurrence stops at rtol; beyond it the true residual holds the
        # rounding of the products: eps |K| |x| over the steps that made up x
        eps = 2.0 ** -24 if prec == _capi.PRECISION_MIXED else 2.0 ** -53
        bound = 1.01 * rtol + 64 * eps * abs(K).sum(axis=1).max() * np.linalg.norm(x) / nb
        return it, res, bound
    finally:
        c.close()


@pytest.mark.parametrize("prec", [_capi.PRECISION_MIXED, _capi.PRECISION_FP64])
@pytest.mark.parametrize("model", list(MODELS))
def test_resident_pcg(monkeypatch, model, prec):
    print(f"[gpu] resident pcg {model} precision {prec}", flush=True)
    rtol = 1e-3 if prec == _capi.PRECISION_MIXED else 1e-10
    it, res, bound = _solve(MODELS[model], prec, rtol)
    assert res <= bound
    monkeypatch.setenv("ONSAS_PCG_RESIDENT", "0")
    itg, resg, bound = _solve(MODELS[model], prec, rtol)
    assert resg <= bound
    assert abs(it - itg) <= 2 + itg // 20  # the same recurrences, other sum orders


@pytest.mark.parametrize("prec", [_capi.PRECISION_MIXED, _capi.PRECISION_FP64])
@pytest.mark.parametrize("model,restart", [
    ("1x1x1", 40), ("4x3x2", 2), ("7x3x3", 40), ("6x4x3", 60), ("6x4x3", 61), ("8x6x3", 17),
    ("10x5x3", 40), ("10x10x10", 40), ("clique 17", 40), ("clique 32", 60), ("clique 33", 40)])
def test_resident_gmres(monkeypatch, model, restart, prec):
    """Restart lengths up to the longest basis it keeps, and one past it."""
    print(f"[gpu] resident gmres({restart}) {model} precision {prec}", flush=True)
    rtol = 1e-3 if prec == _capi.PRECISION_MIXED else 1e-9
    it, res, bound = _solve(MODELS[model], prec, rtol, _capi.LINSOLVE_GMRES, restart)
    assert res <= bound
    monkeypatch.setenv("ONSAS_PCG_RESIDENT", "0")
    itg, resg, bound = _solve(MODELS[model], prec, rtol, _capi.LINSOLVE_GMRES, restart)
    assert resg <= bound
    # a short FP32 restart's count follows the order of its sums (121 to 151 in a
    # host model of 4x3x2 with GMRES(2), over permutations of the unknowns; FP64: 157)
    if prec == _capi.PRECISION_FP64:
        assert abs(it - itg) <= 2 + itg // 20


@pytest.mark.parametrize("kind", [_capi.LINSOLVE_PCG, _capi.LINSOLVE_GMRES])
@pytest.mark.parametrize("prec", [_capi.PRECISION_MIXED, _capi.PRECISION_FP64])
def test_expired_wait_solves_on_the_general_path(monkeypatch, prec, kind):
    """With no patience at all a workgroup that finds a slot not yet written ends
    the launch, and the solve starts again on the general kernels."""
    print(f"[gpu] resident solver {kind}, expired wait, precision {prec}", flush=True)
    rtol = 1e-3 if prec == _capi.PRECISION_MIXED else 1e-10
    monkeypatch.setenv("ONSAS_RESIDENT_TICKS", "-1")
    _, res, bound = _solve(MODELS["10x10x10"], prec, rtol, kind)
    assert res <= bound
