"""Which way the solves of small and mid-size models go (Context.resident_launches): one
workgroup, workgroups met in one XCD or across the device, or the general kernels, at the
sizes where the rules change; and what a launch that gave up leaves behind."""
import numpy as np
import pytest

from onsas_amd import _capi
from test_gpu_resident import MODELS

pytestmark = pytest.mark.gpu

MIXED, FP64 = _capi.PRECISION_MIXED, _capi.PRECISION_FP64
PCG, GMRES = _capi.LINSOLVE_PCG, _capi.LINSOLVE_GMRES


class Solves:
    """Linear solves and Newton steps of one context, and the launches of each."""

    def __init__(self, model, prec, kind, newton=False):
        self.c, nn = MODELS[model](prec)
        self.prec, self.newton = prec, newton
        self.c.set_linear_solver(kind, rtol=1e-3 if prec == MIXED else 1e-8, maxiter=20000)
        self.c.set_U(np.zeros(3 * nn))
        self.b = np.random.default_rng(nn).normal(size=3 * nn)
        self.c.set_loads(nodal=1e-3 * self.b)
        self.c.assemble()

    def __enter__(self):
        return self

    def __exit__(self, *_):
        self.c.close()

    def run(self):
        """(launches by place that this solve added, its solution)"""
        before = self.c.resident_launches()
        if self.newton:
            self.c.assemble()
            self.c.newton_step()
            x = self.c.get_U()
        else:
            x = self.c.linear_solve(self.b)[0]
        after = self.c.resident_launches()
        return {k: n - before[k] for k, n in after.items() if n != before[k]}, x


# (model, precision): where its PCG's workgroups meet, and GMRES(40)'s
PLACES = [
    ("1x1x1", MIXED, "one_workgroup", "one_xcd"), ("1x1x1", FP64, "one_workgroup", "one_xcd"),
    ("7x3x3", FP64, "one_workgroup", "one_xcd"), ("6x4x3", FP64, "one_xcd", "one_xcd"),
    ("8x6x3", MIXED, "one_workgroup", "one_xcd"), ("10x5x3", MIXED, "one_xcd", "one_xcd"),
    ("10x10x10", MIXED, "one_xcd", "one_xcd"), ("10x10x10", FP64, "one_xcd", "one_xcd"),
    ("16x15x15", MIXED, "one_xcd", None), ("16x15x15", FP64, "across_device", None),
    ("21x20x19", MIXED, "across_device", None), ("21x20x19", FP64, "across_device", None),
    ("clique 17", MIXED, "one_workgroup", "one_xcd"), ("clique 32", FP64, "one_workgroup", "one_xcd"),
    ("clique 33", MIXED, "general", "general"), ("clique 33", FP64, "general", "general"),
]


@pytest.mark.parametrize("model,prec,pcg,gmres", PLACES)
def test_where_solves_run(model, prec, pcg, gmres):
    print(f"[gpu] places of {model} precision {prec}", flush=True)
    for kind, place in ((PCG, pcg), (GMRES, gmres)):
        if place is None:  # a restarted GMRES of this size stagnates
            continue
        for newton in (False, True):
            if newton and kind == GMRES and model.startswith("clique"):
                continue
            with Solves(model, prec, kind, newton) as s:
                for _ in range(2):
                    assert s.run()[0] == ({} if place == "general" else {place: 1})


@pytest.mark.parametrize("prec", [MIXED, FP64])
@pytest.mark.parametrize("kind", [PCG, GMRES])
def test_across_the_device_on_request(monkeypatch, prec, kind):
    print(f"[gpu] places across the device, solver {kind} precision {prec}", flush=True)
    monkeypatch.setenv("ONSAS_RESIDENT_XCD", "0")
    with Solves("10x10x10", prec, kind) as s:
        assert s.run()[0] == {"across_device": 1}


@pytest.mark.parametrize("newton", [False, True])
@pytest.mark.parametrize("prec", [MIXED, FP64])
def test_expired_waits_are_counted(monkeypatch, prec, newton):
    """No patience at all: both meeting places are given up in the first solve, which
    then takes the general kernels."""
    print(f"[gpu] expired waits, precision {prec} newton {newton}", flush=True)
    monkeypatch.setenv("ONSAS_RESIDENT_TICKS", "-1")
    with Solves("10x10x10", prec, PCG, newton) as s:
        assert s.run()[0] == {"gave_up": 2}
        assert s.run()[0] == {}


@pytest.mark.parametrize("prec", [MIXED, FP64])
def test_both_meeting_places_give_the_same_bits(monkeypatch, prec):
    """A solve that is taken again across the device adds in the same order."""
    print(f"[gpu] meeting places, precision {prec}", flush=True)
    with Solves("10x10x10", prec, PCG) as s:
        at, x = s.run()
    monkeypatch.setenv("ONSAS_RESIDENT_XCD", "0")
    with Solves("10x10x10", prec, PCG) as s:
        at2, x2 = s.run()
    assert (at, at2) == ({"one_xcd": 1}, {"across_device": 1})
    assert np.array_equal(x, x2)


@pytest.mark.parametrize("kind", [PCG, GMRES])
@pytest.mark.parametrize("prec", [MIXED, FP64])
def test_a_context_comes_back_to_the_fast_path(monkeypatch, prec, kind):
    """Two launches without patience (one XCD, then the device): the context rests for 128
    solves on the general kernels and then stays on the fast path.  With one, it meets across
    the device for 64 solves."""
    print(f"[gpu] coming back, solver {kind} precision {prec}", flush=True)
    for launches, rest, meanwhile in ((2, 128, {}), (1, 64, {"across_device": 1})):
        monkeypatch.setenv("ONSAS_RESIDENT_TICKS", f"-1:{launches}")
        with Solves("10x10x10", prec, kind) as s:
            first = s.run()[0]
            assert first.pop("gave_up") == launches and first == meanwhile
            for _ in range(rest - 1):
                assert s.run()[0] == meanwhile
            for _ in range(2):
                assert s.run()[0] == {"one_xcd": 1}
