"""The work whose speed this framework is judged by: passes through its public
entry points, from a few hundred elements to 1.6 million.

A case is a dict of plain values.  `listed` gives the fixed ones, `draw` others
of the same ranges, `prepare` what a user's program holds before the call (the
model on the GPU, inputs made from the seed), `run` one pass, `work` the bytes
and operations that a pass cannot do without, `exact` the outputs in 64 bits
without the engine.

Kinds:
  newton    a nonlinear static analysis of a box of tetrahedra, solve_ on a model
            that stays on the GPU (as in a parameter study); U of every load step
            and, with `store`, the stresses and strains
  linear    a LinearStaticAnalysis of a thick cylinder under internal pressure
  truss     a nonlinear static analysis of a space-truss lattice
  identify  one step of an identification: new shear moduli, a warm-started
            re-solve, and the gradient of the misfit through the adjoint
  fields    f_int, stresses and strains at a given displacement field
  matvec    a product with the assembled tangent (a caller's own Krylov method)
  locate    point location in the mesh (interpolation of results)
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "onsas.jl_amd"))

from onsas_amd import adjoint, meshes  # noqa: E402
from onsas_amd.analysis import (ConvergenceSettings, NewtonRaphson,  # noqa: E402
                                NonLinearStaticAnalysis, solve, solve_)
from onsas_amd.backend import GpuStaticState, MI355XBackend  # noqa: E402
from onsas_amd.boundary_conditions import (FixedField, GlobalLoad, Pressure,  # noqa: E402
                                           StructuralBoundaryCondition)
from onsas_amd.entities import (Circle, Mesh, NodeSet, RotatedEngineeringStrain,  # noqa: E402
                                Tetrahedra, TriangularFaces, Trusses)
from onsas_amd.linear_analysis import LinearStaticAnalysis  # noqa: E402
from onsas_amd.materials import IsotropicLinearElastic, NeoHookean, SVK  # noqa: E402
from onsas_amd.structure import StructuralMaterial, Structure  # noqa: E402

NH_K, NH_G = 8.3e5, 3.8e5  # the uniaxial compression example's bulk and shear moduli
SVK_E, SVK_NU = 1e6, 0.3   # the uniaxial extension example's
CYL_E, CYL_NU = 210e9, 0.3
DENSE = 9000  # most dofs that exact() solves with a dense matrix


def _newton(name, nx, ny, nz, mat, prec, solver, steps, store=True, forcing=False,
            refresh="step"):
    c = dict(kind="newton", nx=nx, ny=ny, nz=nz, mat=mat, prec=prec, solver=solver, steps=steps,
             store=store, forcing=forcing, refresh=refresh)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the examples' own scale: every default of the backend, stresses stored per load step
        _newton("newton 4x4x4 svk", 4, 4, 4, "svk", "mixed", "jacobi", 8),
        # a part meshed coarsely, sides that divide nothing; default backend
        _newton("newton 13x9x11 nh", 13, 9, 11, "nh", "mixed", "jacobi", 4),
        # the GMRES solver option (indefinite tangents need it), the reference's precision
        _newton("newton 9x8x7 gmres", 9, 8, 7, "svk", "fp64", "gmres", 2),
        # multigrid with its default refresh (each load step), all FP64, stresses stored
        _newton("newton 23x17x19 amg fp64", 23, 17, 19, "nh", "fp64", "amg", 3),
        # the benchmark's compression cube and settings: 1.57 M tetrahedra, 20 load steps
        _newton("newton 64x64x64 amg", 64, 64, 64, "nh", "mixed", "amg", 20, store=False,
                forcing=True, refresh="once"),
        # linear elasticity, FP64, block-Jacobi: the cylinder example's scale
        dict(name="linear 4x32x12", kind="linear", nr=4, nt=32, nz=12, prec="fp64",
             solver="jacobi", steps=2),
        # linear elasticity at an engineering mesh size, mixed precision with refinement
        dict(name="linear 12x96x48 amg", kind="linear", nr=12, nt=96, nz=48, prec="mixed",
             solver="amg", steps=2),
        # space truss (two-node bars, nodal loads)
        dict(name="truss 11", kind="truss", n=11, prec="mixed", solver="jacobi", steps=4),
        # gradient-based identification of a stiffness field
        dict(name="identify 24x24x24", kind="identify", nx=24, ny=24, nz=24, prec="mixed",
             solver="amg"),
        # recovery of forces and stresses of a state (post-processing, explicit updates)
        dict(name="fields 48x31x37", kind="fields", nx=48, ny=31, nz=37, mat="nh", prec="mixed"),
        # the tangent as a linear operator of a caller's solver
        dict(name="matvec 37x33x29", kind="matvec", nx=37, ny=33, nz=29, mat="svk", prec="fp64"),
        # evaluation of results at points
        dict(name="locate 100k", kind="locate", nx=32, ny=29, nz=35, points=100003),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _sides(rng, lo, hi):
    """Three sides around one log-spread size."""
    m = lo * (hi / lo) ** rng.random()
    return [max(2, min(hi, int(round(m * rng.uniform(0.75, 1.3))))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["newton"] * 5 + ["linear", "linear", "truss", "identify", "fields",
                                        "matvec", "locate"])
    prec = rng.choice(["mixed", "fp64"])
    if kind == "newton":
        solver = rng.choice(["jacobi", "jacobi", "amg", "amg", "gmres"])
        nx, ny, nz = _sides(rng, 3, {"jacobi": 22, "amg": 48, "gmres": 8}[solver])
        if solver == "gmres":
            prec = "fp64"
        return _newton(None, nx, ny, nz, rng.choice(["svk", "nh"]), prec, solver,
                       rng.randint(2, 6) if solver != "gmres" else 2,
                       store=nx * ny * nz < 12000 and rng.random() < 0.7,
                       forcing=solver == "amg" and rng.random() < 0.5,
                       refresh=rng.choice(["step", "once"]))
    if kind == "linear":
        solver = rng.choice(["jacobi", "amg"])
        m = _log_int(rng, 3, 6 if solver == "jacobi" else 14)
        return dict(kind=kind, nr=m, nt=4 * rng.randint(max(4, m), 2 * max(4, m)),
                    nz=rng.randint(2 * m, 4 * m), prec=prec, solver=solver, steps=rng.randint(1, 3))
    if kind == "truss":
        return dict(kind=kind, n=_log_int(rng, 3, 16), prec=prec,
                    solver=rng.choice(["jacobi", "amg"]), steps=rng.randint(2, 5))
    if kind == "locate":
        nx, ny, nz = _sides(rng, 4, 36)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, points=_log_int(rng, 50, 200000))
    nx, ny, nz = _sides(rng, 4, 28 if kind == "identify" else 48)
    c = dict(kind=kind, nx=nx, ny=ny, nz=nz, prec=prec)
    if kind == "identify":
        return dict(c, solver="amg" if nx * ny * nz > 4000 else rng.choice(["jacobi", "amg"]))
    return dict(c, mat=rng.choice(["svk", "nh"]), prec="fp64" if kind == "matvec" else prec)


# ---- models ----------------------------------------------------------------------

def _box(case, seed):
    """Unit cube of nx x ny x nz cells x 6 tetrahedra, interior nodes moved by up
    to 3 % of the cell (affine fields stay exact)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    sm = meshes.cube(nx, ny=ny, nz=nz)
    X = sm.coords
    inner = np.all((X > 1e-12) & (X < 1 - 1e-12), axis=1)
    r = np.random.default_rng([seed, 1]).uniform(-0.03, 0.03, size=X.shape)
    X[inner] += r[inner] / np.array([nx, ny, nz])
    return sm


def _alpha(seed):
    """Final stretch of the compression (a seeded load level)."""
    return 0.85 + 0.03 * float(np.random.default_rng([seed, 2]).uniform(-1, 1))


def _tension(seed):
    return 3e5 * (1 + 0.1 * float(np.random.default_rng([seed, 2]).uniform(-1, 1)))


def _nh_p11(a):
    """Nominal stress and squared lateral stretch of uniaxial NeoHookean at stretch a."""
    b = 1.0
    for _ in range(100):
        f = NH_G * (b - 1 / b) + NH_K * b * (a * a * b * b - a)
        b -= f / (NH_G * (1 + 1 / b ** 2) + NH_K * (3 * a * a * b * b - a))
    return NH_G * (a - 1 / a) + NH_K * b * b * (a * b * b - 1), b


def _nh_alpha(p11):
    a = 1.0
    for _ in range(100):
        h = 1e-6
        a -= (_nh_p11(a)[0] - p11) / ((_nh_p11(a + h)[0] - _nh_p11(a - h)[0]) / (2 * h))
    return a


def _svk_alpha(p):
    a = 1.0
    for _ in range(100):
        a -= (SVK_E / 2 * a * (a * a - 1) - p) / (SVK_E / 2 * (3 * a * a - 1))
    return a


def _material(mat, G=None):
    if mat == "svk":
        return SVK(E=SVK_E, nu=SVK_NU, label="mat")
    return NeoHookean(NH_K, NH_G if G is None else G, label="mat")


def _load(mat, seed):
    return -_tension(seed) if mat == "svk" else -_nh_p11(_alpha(seed))[0]


def _box_structure(case, seed, G=None):
    """Rollers on x = 0, y = 0, z = 0; pressure p t on x = 1."""
    sm = _box(case, seed)
    mat = case.get("mat", "nh")
    tets = Tetrahedra(sm.tets, "tets")
    faces = {k: TriangularFaces(f, k) for k, f in sm.faces.items()}
    p = _load(mat, seed)
    bcs = {FixedField("u", [1], "ux"): [faces["x0"]], FixedField("u", [2], "uy"): [faces["y0"]],
           FixedField("u", [3], "uz"): [faces["z0"]],
           Pressure("u", lambda t: p * t, "p"): [faces["x1"]]}
    s = Structure(Mesh(sm.coords, [tets], list(faces.values())),
                  StructuralMaterial({_material(mat, G): tets}), StructuralBoundaryCondition(bcs))
    return s, sm


def _backend(case):
    solver = case.get("solver", "jacobi")
    return MI355XBackend(
        precision=case["prec"], maxiter=20000, solver="gmres" if solver == "gmres" else "auto",
        preconditioner="amg" if solver == "amg" else "block-jacobi",
        amg_refresh=case.get("refresh", "step"), forcing=case.get("forcing", False),
        store_stresses=case.get("store", case["kind"] == "linear"),
        rtol=1e-12 if case["kind"] == "linear" and case["prec"] == "fp64" else None)


def _newton_alg():
    # the tighter of the test-suite's tolerances: results then hold to about 1e-10
    return NewtonRaphson(ConvergenceSettings(rel_U_tol=1e-14, rel_res_force_tol=1e-10, max_iter=30))


def _identify_alg():
    return NewtonRaphson(ConvergenceSettings(rel_U_tol=1e-16, rel_res_force_tol=1e-12, max_iter=40))


def _moduli(sm, seed):
    """A smooth random shear-modulus field, one value per element."""
    r = np.random.default_rng([seed, 3])
    w, phi = r.normal(size=(24, 3)) / 0.3, r.uniform(0, 2 * np.pi, 24)
    cen = sm.coords[sm.tets].mean(axis=1)
    return NH_G * np.exp(0.2 * np.sqrt(2 / 24) * np.cos(cen @ w.T + phi).sum(axis=1))


def _displacement(sm, seed):
    """A finite deformation: a stretch plus smooth waves (strains of a few percent)."""
    r = np.random.default_rng([seed, 4])
    A = 0.03 * r.normal(size=(3, 3))
    k, ph, amp = r.integers(1, 4, (3, 3)), r.uniform(0, 2 * np.pi, (3, 3)), 0.004 * r.normal(size=(3, 3))
    X = sm.coords
    u = X @ A.T
    for d in range(3):
        for q in range(3):
            u[:, d] += amp[d, q] * np.sin(2 * np.pi * k[d, q] * X[:, q] + ph[d, q])
    return u.reshape(-1)


def _cylinder(case, seed):
    r = np.random.default_rng([seed, 5])
    Ri, Re, p = 0.1 * (1 + 0.05 * r.uniform(-1, 1)), 0.2, 1e7 * (1 + 0.1 * r.uniform(-1, 1))
    sm = meshes.cylinder(case["nr"], case["nt"], case["nz"], Ri, Re, 0.5)
    return sm, p


def _cylinder_structure(case, seed):
    sm, p = _cylinder(case, seed)
    tets, inner = Tetrahedra(sm.tets, "tets"), TriangularFaces(sm.faces["inner"], "inner")
    bcs = {FixedField("u", [3], "uz"): [NodeSet(np.concatenate([sm.node_sets["z0"],
                                                                sm.node_sets["z1"]]))],
           FixedField("u", [2], "uy"): [NodeSet(sm.node_sets["theta0"])],
           FixedField("u", [1], "ux"): [NodeSet(sm.node_sets["theta90"])],
           Pressure("u", lambda t: p * t, "p"): [inner]}
    return Structure(Mesh(sm.coords, [tets], [inner]),
                     StructuralMaterial({IsotropicLinearElastic(CYL_E, CYL_NU, "mat"): tets}),
                     StructuralBoundaryCondition(bcs)), sm


TR_H, TR_A = 0.1, 1e-4  # lattice spacing and bar area of the truss workload


def _lattice(case, seed):
    sm = meshes.truss_lattice(case["n"], h=TR_H, jitter=0.01, seed=seed & 0xffff)
    F = -3e4 * (1 + 0.1 * float(np.random.default_rng([seed, 6]).uniform(-1, 1)))
    return sm, F


def _truss_structure(case, seed):
    sm, F = _lattice(case, seed)
    bars = Trusses(sm.trusses, Circle(float(np.sqrt(4 * TR_A / np.pi))), RotatedEngineeringStrain,
                   "bars")
    bcs = {FixedField("u", [1, 2, 3], "pin"): [NodeSet(sm.node_sets["z0"])],
           GlobalLoad("u", lambda t: [0.0, 0.0, F * t], "top"): [NodeSet(sm.node_sets["z1"])]}
    return Structure(Mesh(sm.coords, [bars]),
                     StructuralMaterial({SVK(E=CYL_E, nu=CYL_NU, label="mat"): bars}),
                     StructuralBoundaryCondition(bcs))


def _points(case, sm, seed):
    """Points inside known elements, about a tenth of them outside the mesh."""
    r = np.random.default_rng([seed, 7])
    n = case["points"]
    e = r.integers(0, len(sm.tets), n)
    w = 0.02 + 0.92 * r.dirichlet([1, 1, 1, 1], n)
    P = np.einsum("pa,pad->pd", w, sm.coords[sm.tets[e]])
    out = r.random(n) < 0.1
    P[out] += 1.5
    return P, np.where(out, -1, e).astype(np.int64), np.where(out[:, None], 0.0, w)


# ---- the interface ---------------------------------------------------------------

def prepare(case, seed):
    k, st = case["kind"], {"case": case}
    if k == "truss":
        s = _truss_structure(case, seed)
    elif k == "linear":
        s, _ = _cylinder_structure(case, seed)
    else:
        G = None
        if k == "identify":
            G = np.full(6 * case["nx"] * case["ny"] * case["nz"], NH_G)
        s, sm = _box_structure(case, seed, G)
    if k == "identify":
        # the start of the identification: a uniform guess, solved
        sa = NonLinearStaticAnalysis(s, NSTEPS=2)
        st["backend"], st["alg"] = _backend(case), _identify_alg()
        st["sol"], st["pullback"] = adjoint.rrule(solve, sa, st["alg"], st["backend"])
        st["G"] = _moduli(sm, seed)
        r = np.random.default_rng([seed, 8])
        surf = np.unique(np.concatenate([sm.node_sets[q] for q in ("x1", "y1", "z1")]))
        st["obs"] = np.sort(r.choice(surf, size=min(2000, len(surf)), replace=False))
        U = st["sol"].U[-1].reshape(-1, 3)[st["obs"]]
        st["target"] = U * (1 + 0.05 * r.normal(size=U.shape))
        return st
    if k == "locate":
        st["gpu"] = GpuStaticState(s, MI355XBackend())
        st["points"] = _points(case, sm, seed)[0]
        return st
    st["s"], st["backend"] = s, _backend(case)
    st["gpu"] = GpuStaticState(s, st["backend"])
    if k in ("newton", "truss"):
        st["alg"], st["zeros"] = _newton_alg(), np.zeros(s.num_dofs())
    elif k == "fields":
        st["U"] = _displacement(sm, seed)
    elif k == "matvec":
        st["gpu"].ctx.set_U(_displacement(sm, seed))
        st["gpu"].ctx.assemble()
        st["x"] = np.random.default_rng([seed, 9]).normal(size=s.num_dofs())
    return st


def run(st):
    case = st["case"]
    k = case["kind"]
    if k in ("newton", "truss"):
        sa = NonLinearStaticAnalysis(st["s"], NSTEPS=case["steps"], initial_state=st["zeros"])
        sa.state = st["gpu"]
        sol = solve_(sa, st["alg"], st["backend"])
        return _solution(sol, st["backend"].store_stresses)
    if k == "linear":
        sa = LinearStaticAnalysis(st["s"], NSTEPS=case["steps"])
        sa.state = st["gpu"]
        return _solution(solve_(sa, None, st["backend"]), True)
    if k == "identify":
        sol = adjoint.resolve(st["sol"], st["G"], st["alg"], st["backend"])
        J, g = adjoint.misfit(sol.U[-1], st["obs"], st["target"])
        return {"J": J, "U": sol.U[-1], "grad": st["pullback"](g)["tets"]}
    ctx = st["gpu"].ctx
    if k == "fields":
        ctx.set_U(st["U"])
        f = ctx.assemble(want_fint=True)
        stress, strain = ctx.stress_strain(0)
        return {"f": f, "stress": stress, "strain": strain}
    if k == "matvec":
        return ctx.matvec(st["x"])
    return list(ctx.locate_points(0, st["points"]))


def _solution(sol, store):
    out = {"U": list(sol.U)}
    if store:
        out["stress"] = [s[0] for s in sol.stress]
        out["strain"] = [s[0] for s in sol.strain]
    return out


def work(case):
    """Counts of what a pass cannot do without.  Elements: connectivity and
    nodal state in, tangent blocks (15 per node of these meshes) out, about 700
    operations per tetrahedron.  Iterative solves: one pass over the tangent and
    five vectors per iteration, with the iterations that the preconditioner
    takes on such meshes (block-Jacobi: a few per element layer; multigrid:
    five, each with two more passes over the tangent)."""
    k = case["kind"]
    if k == "truss":
        nn, ne = (case["n"] + 1) ** 3, 7 * case["n"] ** 3
        layers = case["n"]
    elif k == "linear":
        nn = (case["nr"] + 1) * case["nt"] * (case["nz"] + 1)
        ne = 6 * case["nr"] * case["nt"] * case["nz"]
        layers = max(case["nt"] // 2, case["nz"])
    else:
        nn = (case["nx"] + 1) * (case["ny"] + 1) * (case["nz"] + 1)
        ne = 6 * case["nx"] * case["ny"] * case["nz"]
        layers = max(case["nx"], case["ny"], case["nz"])
    kt = 8 if case.get("prec") == "fp64" else 4
    tangent = 15 * nn * (9 * kt + 4)
    asm = ne * 16 + 48 * nn + tangent
    stress = 2 * 72 * ne
    if k == "locate":
        return {"bytes": case["points"] * 64.0, "flops": case["points"] * 60.0}
    if k == "fields":
        return {"bytes": 48.0 * nn + 16 * ne + stress, "flops": 400.0 * ne}
    if k == "matvec":
        return {"bytes": tangent + 48.0 * nn, "flops": 18.0 * 15 * nn}
    amg = case["solver"] == "amg"
    passes = 5 * 3 if amg else 3 * layers
    solve_b = passes * (tangent + 15 * nn * kt)
    solve_f = passes * 18 * 15 * nn
    newtons = {"newton": 4, "truss": 3, "linear": 1, "identify": 5}[k] * case.get("steps", 1)
    stores = case.get("steps", 1) * (24 * nn + (stress if case.get("store", k == "linear") else 0))
    return {"bytes": float(newtons * (asm + solve_b) + stores),
            "flops": float(newtons * (700 * ne + solve_f))}


# ---- 64-bit values without the engine ---------------------------------------------

def exact(case, seed):
    k = case["kind"]
    if k == "newton":
        return _exact_uniaxial(case, seed)
    if k == "locate":
        return list(_points(case, _box(case, seed), seed)[1:])
    if k in ("fields", "matvec"):
        sm = _box(case, seed)
        U = _displacement(sm, seed).reshape(-1, 3)
        if k == "fields":
            f, P, C = _tet_state(sm, U, case["mat"])
            return {"f": f, "stress": P, "strain": C}
        x = np.random.default_rng([seed, 9]).normal(size=3 * sm.nn)
        return _tangent_product(sm, U, case["mat"], x)
    if k == "linear":
        return _exact_linear(case, seed)
    if k == "truss":
        return _exact_truss(case, seed)
    return None  # identify: a nonlinear solve and an adjoint of tens of thousands of dofs


def _exact_uniaxial(case, seed):
    """The uniaxial closed forms (homogeneous states)."""
    sm = _box(case, seed)
    out = {"U": [], "stress": [], "strain": []}
    for t in np.linspace(1 / case["steps"], 1, case["steps"]):
        if case["mat"] == "svk":
            p = _tension(seed) * t
            a = _svk_alpha(p)
            b = np.sqrt(1 - SVK_NU * (a * a - 1))
        else:
            p = -_load("nh", seed) * t
            a = _nh_alpha(p)
            b = _nh_p11(a)[1]
        out["U"].append(((np.array([a, b, b]) - 1) * sm.coords).reshape(-1))
        if case["store"]:
            one = np.ones((len(sm.tets), 1, 1))
            out["stress"].append(one * np.diag([p, 0.0, 0.0]))
            out["strain"].append(one * np.diag([a * a, b * b, b * b]))
    return out if case["store"] else {"U": out["U"]}


def _gradients(X, tets):
    """Shape-function gradients (ne, 4, 3) and volumes."""
    x = X[tets]
    J = x[:, 1:] - x[:, :1]                   # rows X_a - X_0
    g = np.linalg.inv(J).transpose(0, 2, 1)   # rows grad N_1..3
    n = np.concatenate([-g.sum(axis=1, keepdims=True), g], axis=1)
    return n, np.abs(np.linalg.det(J)) / 6


def _second_pk(F, mat):
    I3 = np.eye(3)
    C = F.transpose(0, 2, 1) @ F
    if mat == "svk":
        lam, G = SVK_E * SVK_NU / ((1 + SVK_NU) * (1 - 2 * SVK_NU)), SVK_E / (2 * (1 + SVK_NU))
        E = 0.5 * (C - I3)
        return C, lam * np.trace(E, axis1=1, axis2=2)[:, None, None] * I3 + 2 * G * E
    Ci = np.linalg.inv(C)
    J = np.sqrt(np.linalg.det(C))[:, None, None]
    return C, NH_G * (I3 - Ci) + NH_K * J * (J - 1) * Ci


def _scatter(sm, fe):
    f = np.zeros((sm.nn, 3))
    for d in range(3):
        f[:, d] = np.bincount(sm.tets.reshape(-1), fe[:, :, d].reshape(-1), sm.nn)
    return f


def _tet_state(sm, U, mat):
    n, V = _gradients(sm.coords, sm.tets)
    F = np.eye(3) + U[sm.tets].transpose(0, 2, 1) @ n
    C, S = _second_pk(F, mat)
    P = F @ S
    return _scatter(sm, V[:, None, None] * (n @ P.transpose(0, 2, 1))).reshape(-1), P, C


def _tangent_product(sm, U, mat, x):
    """K x with unit rows and columns at the rollers: the directional derivative of f."""
    fixed = np.zeros((sm.nn, 3), bool)
    for d, q in enumerate(("x0", "y0", "z0")):
        fixed[sm.node_sets[q], d] = True
    x = x.reshape(-1, 3)
    n, V = _gradients(sm.coords, sm.tets)
    F = np.eye(3) + U[sm.tets].transpose(0, 2, 1) @ n
    dF = np.where(fixed, 0.0, x)[sm.tets].transpose(0, 2, 1) @ n
    C, S = _second_pk(F, mat)
    dC = dF.transpose(0, 2, 1) @ F + F.transpose(0, 2, 1) @ dF
    if mat == "svk":
        lam, G = SVK_E * SVK_NU / ((1 + SVK_NU) * (1 - 2 * SVK_NU)), SVK_E / (2 * (1 + SVK_NU))
        dS = 0.5 * lam * np.trace(dC, axis1=1, axis2=2)[:, None, None] * np.eye(3) + G * dC
    else:
        Ci = np.linalg.inv(C)
        J = np.sqrt(np.linalg.det(C))[:, None, None]
        dCi = -Ci @ dC @ Ci
        dJ = 0.5 * J * np.trace(Ci @ dC, axis1=1, axis2=2)[:, None, None]
        dS = -NH_G * dCi + NH_K * ((2 * J - 1) * dJ * Ci + J * (J - 1) * dCi)
    dP = dF @ S + F @ dS
    y = _scatter(sm, V[:, None, None] * (n @ dP.transpose(0, 2, 1)))
    return np.where(fixed, x, y).reshape(-1)


def _dense_solve(K, b):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    return torch.linalg.solve(K.to(dev), torch.from_numpy(b).to(dev)).cpu().numpy()


def _exact_linear(case, seed):
    sm, p = _cylinder(case, seed)
    n3 = 3 * sm.nn
    if n3 > DENSE:
        return None
    n, V = _gradients(sm.coords, sm.tets)
    lam, G = CYL_E * CYL_NU / ((1 + CYL_NU) * (1 - 2 * CYL_NU)), CYL_E / (2 * (1 + CYL_NU))
    nn = np.einsum("eai,ebj->eabij", n, n)
    Ke = (lam * nn + G * nn.transpose(0, 1, 2, 4, 3)
          + G * np.einsum("eab,ij->eabij", n @ n.transpose(0, 2, 1), np.eye(3)))
    Ke = (V[:, None, None, None, None] * Ke).transpose(0, 1, 3, 2, 4).reshape(-1, 12, 12)
    dofs = (3 * sm.tets[:, :, None].astype(np.int64) + np.arange(3)).reshape(-1, 12)
    K = torch.zeros(n3 * n3, dtype=torch.float64)
    K.index_add_(0, torch.from_numpy((dofs[:, :, None] * n3 + dofs[:, None, :]).reshape(-1)),
                 torch.from_numpy(Ke.reshape(-1)))
    fixed = np.zeros((sm.nn, 3), bool)
    fixed[sm.node_sets["z0"], 2] = fixed[sm.node_sets["z1"], 2] = True
    fixed[sm.node_sets["theta0"], 1] = fixed[sm.node_sets["theta90"], 0] = True
    free = np.nonzero(~fixed.reshape(-1))[0]
    tri = sm.faces["inner"]
    x = sm.coords[tri]
    av = 0.5 * np.cross(x[:, 1] - x[:, 0], x[:, 2] - x[:, 0])
    f = np.zeros((sm.nn, 3))
    for a in range(3):
        np.add.at(f, tri[:, a], -p * av / 3)
    ft = torch.from_numpy(free)
    Kff = K.view(n3, n3).index_select(0, ft).index_select(1, ft)
    U1 = np.zeros(n3)
    U1[free] = _dense_solve(Kff, f.reshape(-1)[free])
    H = U1.reshape(-1, 3)[sm.tets].transpose(0, 2, 1) @ n
    eps = 0.5 * (H + H.transpose(0, 2, 1))
    sig = lam * np.trace(eps, axis1=1, axis2=2)[:, None, None] * np.eye(3) + 2 * G * eps
    ts = np.linspace(1 / case["steps"], 1, case["steps"])
    return {"U": [t * U1 for t in ts], "stress": [t * sig for t in ts],
            "strain": [t * eps for t in ts]}


def _exact_truss(case, seed):
    sm, F = _lattice(case, seed)
    n3 = 3 * sm.nn
    if n3 > DENSE:
        return None
    i, j = sm.trusses[:, 0], sm.trusses[:, 1]
    D = sm.coords[j] - sm.coords[i]
    l0 = np.linalg.norm(D, axis=1)
    fixed = np.zeros((sm.nn, 3), bool)
    fixed[sm.node_sets["z0"]] = True
    free = np.nonzero(~fixed.reshape(-1))[0]
    ft = torch.from_numpy(free)
    load = np.zeros((sm.nn, 3))
    load[sm.node_sets["z1"], 2] = F
    da, db = (3 * q[:, None].astype(np.int64) + np.arange(3) for q in (i, j))
    U, out = np.zeros(n3), []
    for t in np.linspace(1 / case["steps"], 1, case["steps"]):
        for _ in range(8):
            u = U.reshape(-1, 3)
            du = u[j] - u[i]
            d = D + du
            l = np.linalg.norm(d, axis=1)
            # (l^2 - l0^2) / (l0 (l0 + l)) without cancellation
            N = CYL_E * TR_A * (2 * (D * du).sum(1) + (du * du).sum(1)) / (l0 * (l0 + l))
            e = d / l[:, None]
            fi = np.zeros((sm.nn, 3))
            np.add.at(fi, j, N[:, None] * e)
            np.add.at(fi, i, -N[:, None] * e)
            r = (t * load - fi).reshape(-1)[free]
            if np.linalg.norm(r) <= 1e-13 * np.linalg.norm(t * load):
                break
            k3 = ((N / l)[:, None, None] * np.eye(3)
                  + (CYL_E * TR_A / l0 - N / l)[:, None, None] * e[:, :, None] * e[:, None, :])
            K = torch.zeros(n3 * n3, dtype=torch.float64)
            for a, b, s in ((da, da, 1), (db, db, 1), (da, db, -1), (db, da, -1)):
                K.index_add_(0, torch.from_numpy((a[:, :, None] * n3 + b[:, None, :]).reshape(-1)),
                             torch.from_numpy(s * k3.reshape(-1)))
            U[free] += _dense_solve(K.view(n3, n3).index_select(0, ft).index_select(1, ft), r)
        out.append(U.copy())
    return {"U": out}
