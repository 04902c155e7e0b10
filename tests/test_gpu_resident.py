"""The one-launch block-Jacobi PCG and GMRES of small models (resident_solve.hip) at the
edges of its shapes: one workgroup and several, full and partial ones, 4 and 8
lanes a row, models just past its limits, and the path a launch takes when a
wait for the other workgroups expires."""
import numpy as np
import pytest
from scipy.sparse.linalg import eigsh

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


def _newton_run(make, prec, forcing=False, kind=_capi.LINSOLVE_AUTO, steps=2, its=6):
    """`steps` load steps of `its` Newton iterations (the later steps start warm): U after
    every iteration, the statistics and the last tangent on the free dofs."""
    c, nn = make(prec)
    try:
        c.set_linear_solver(kind, rtol=1e-6 if prec == _capi.PRECISION_MIXED else 1e-10,
                            maxiter=20000, forcing=forcing, newton_tol=1e-8 if forcing else 0.0)
        f = np.zeros((nn, 3))
        f[:, 0], f[:, 2] = 4e3 / nn, -2e3 / nn
        c.set_U(np.zeros(3 * nn))
        Us, log = [], []
        for s in range(steps):
            c.set_loads(nodal=(s + 1.0) * f.reshape(-1))
            for _ in range(its):
                c.assemble()
                log.append(c.newton_step())
                Us.append(c.get_U())
        fnorm = np.linalg.norm(c.get_fext())
        c.assemble()
        K = c.tangent_bsr().tocsr()
        free = np.flatnonzero(np.asarray(abs(K).sum(axis=1)).ravel() != 1)
        K = K[free][:, free].tocsc()
        return Us, log, K, fnorm
    finally:
        c.close()


def _stat(st, name):
    return st[name] if isinstance(st, dict) else getattr(st, name)


def _compare_newton(make, prec, monkeypatch, forcing=False, solver=1):
    its = 6 if not forcing else 9
    U, log, K, fn = _newton_run(make, prec, forcing, its=its)
    monkeypatch.setenv("ONSAS_PCG_RESIDENT", "0")
    Ug, logg, _, _ = _newton_run(make, prec, forcing, its=its)
    first, firstg = log[0], logg[0]
    for name in ("r_norm", "fext_norm", "U_norm"):  # of the same data, in another order
        assert np.isclose(_stat(first, name), _stat(firstg, name), rtol=1e-12, atol=0)
    for s in (log, logg):
        assert all(_stat(d, "lin_solver") == solver for d in s)
    # both end within eps of their last residuals' preimage: |U - U'| <= (|r| + |r'|) / smin(K)
    lam = abs(eigsh(K, k=1, sigma=0, return_eigenvectors=False)[0])
    for k in (its - 1, 2 * its - 1):
        r, rg = _stat(log[k], "r_norm"), _stat(logg[k], "r_norm")
        assert r <= 1e-6 * fn and rg <= 1e-6 * fn
        assert np.linalg.norm(U[k] - Ug[k]) <= 2 * (r + rg) / lam + 1e-12 * np.linalg.norm(Ug[k])
    return log, logg


@pytest.mark.parametrize("forcing", [False, True])
@pytest.mark.parametrize("prec", [_capi.PRECISION_MIXED, _capi.PRECISION_FP64])
@pytest.mark.parametrize("model", ["1x1x1", "4x3x2", "6x4x3", "10x5x3", "10x10x10"])
def test_resident_newton_step(monkeypatch, model, prec, forcing):
    """The one-launch Newton step against the step launch by launch."""
    print(f"[gpu] resident newton {model} precision {prec} forcing {forcing}", flush=True)
    log, logg = _compare_newton(MODELS[model], prec, monkeypatch, forcing)
    assert abs(_stat(log[0], "lin_iters") - _stat(logg[0], "lin_iters")) <= \
        2 + _stat(logg[0], "lin_iters") // 20


@pytest.mark.parametrize("prec", [_capi.PRECISION_MIXED, _capi.PRECISION_FP64])
def test_resident_newton_breakdown(monkeypatch, prec):
    """A negative definite tangent: PCG breaks down inside the launch, GMRES takes over."""
    print(f"[gpu] resident newton, breakdown, precision {prec}", flush=True)

    def make(p):
        sm = meshes.cube(4, ny=3, nz=2, jitter=0.05, seed=4)
        c = Context(p)
        c.set_nodes(sm.coords)
        c.add_tet_group(sm.tets, _capi.MAT_NEOHOOKEAN, (-8.3e5, -3.8e5))
        c.set_fixed_dofs((3 * sm.node_sets["x0"][:, None] + np.arange(3)).reshape(-1))
        c.finalize()
        return c, sm.nn

    _compare_newton(make, prec, monkeypatch, solver=3)


@pytest.mark.parametrize("prec", [_capi.PRECISION_MIXED, _capi.PRECISION_FP64])
def test_resident_newton_expired_wait(monkeypatch, prec):
    """A step whose launch gave up is taken again from the state before it, bit for bit."""
    print(f"[gpu] resident newton, expired wait, precision {prec}", flush=True)
    monkeypatch.setenv("ONSAS_RESIDENT_TICKS", "-1")
    U, log, _, _ = _newton_run(MODELS["10x10x10"], prec, forcing=True, its=3)
    monkeypatch.setenv("ONSAS_PCG_RESIDENT", "0")
    Ug, logg, _, _ = _newton_run(MODELS["10x10x10"], prec, forcing=True, its=3)
    for a, b in zip(U, Ug):
        assert np.array_equal(a, b)
    for a, b in zip(log, logg):
        assert _stat(a, "r_norm") == _stat(b, "r_norm")
        assert _stat(a, "lin_iters") == _stat(b, "lin_iters")


@pytest.mark.parametrize("kind", [_capi.LINSOLVE_PCG, _capi.LINSOLVE_GMRES])
@pytest.mark.parametrize("prec", [_capi.PRECISION_MIXED, _capi.PRECISION_FP64])
@pytest.mark.parametrize("model", ["8x6x3", "10x10x10", "16x15x15", "21x20x19"])
def test_resident_across_the_device(monkeypatch, model, prec, kind):
    """The same solves by workgroups that meet in device memory, not in one XCD's L2
    (the only way of the largest model, whose workgroups one XCD does not hold)."""
    print(f"[gpu] resident solver {kind} {model} precision {prec}, across the device", flush=True)
    rtol = 1e-3 if prec == _capi.PRECISION_MIXED else 1e-10
    if kind == _capi.LINSOLVE_GMRES:
        if model in ("16x15x15", "21x20x19"):
            pytest.skip("a restarted GMRES of this size stagnates on either path")
        rtol = max(rtol, 1e-9)
    it, res, bound = _solve(MODELS[model], prec, rtol, kind)
    assert res <= bound
    monkeypatch.setenv("ONSAS_RESIDENT_XCD", "0")
    itd, resd, bound = _solve(MODELS[model], prec, rtol, kind)
    assert resd <= bound
    assert abs(it - itd) <= 2 + itd // 20


def test_resident_contexts_at_the_same_time():
    """Ten contexts solving on threads of their own (more than there are XCDs): whichever
    way a solve ends up taking, it meets its bound."""
    from concurrent.futures import ThreadPoolExecutor
    print("[gpu] resident solves of ten contexts at a time", flush=True)
    kinds = [(_capi.PRECISION_FP64, 1e-10), (_capi.PRECISION_MIXED, 1e-3)]
    with ThreadPoolExecutor(10) as pool:
        runs = [pool.submit(_solve, MODELS["16x15x15" if i % 3 else "10x10x10"], *kinds[i % 2])
                for i in range(10)]
        for f in runs:
            _, res, bound = f.result()
            assert res <= bound


@pytest.mark.parametrize("prec", [_capi.PRECISION_MIXED, _capi.PRECISION_FP64])
def test_resident_newton_breakdown_across_workgroups(monkeypatch, prec):
    """PCG only on a negative definite tangent of many workgroups, with forcing: every one
    of them leaves the first iteration the same way, the step is an error as on the
    general path, and U stays."""
    print(f"[gpu] resident newton, breakdown of many workgroups, precision {prec}", flush=True)
    sm = meshes.cube(10, jitter=0.05, seed=4)
    for resident in ("1", "0"):
        monkeypatch.setenv("ONSAS_PCG_RESIDENT", resident)
        c = Context(prec)
        try:
            c.set_nodes(sm.coords)
            c.add_tet_group(sm.tets, _capi.MAT_NEOHOOKEAN, (-8.3e5, -3.8e5))
            c.set_fixed_dofs((3 * sm.node_sets["x0"][:, None] + np.arange(3)).reshape(-1))
            c.finalize()
            c.set_linear_solver(_capi.LINSOLVE_PCG, rtol=1e-6, maxiter=20000, forcing=True,
                                newton_tol=1e-8)
            U = 1e-3 * np.random.default_rng(1).normal(size=3 * sm.nn)
            f = np.ones(3 * sm.nn)
            for _ in range(3):
                c.set_U(U)
                c.set_loads(nodal=f)
                c.assemble()
                with pytest.raises(_capi.OnsasError, match="breakdown"):
                    c.newton_step()
                assert np.array_equal(c.get_U(), U)
        finally:
            c.close()
