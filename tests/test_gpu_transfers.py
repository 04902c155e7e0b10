"""Per-element results on both sides of the size above which they come back through
the pinned ring, with whole and partial chunks: every element's stress and strain
in its place."""
import numpy as np
import pytest

from onsas_amd import _capi, meshes
from onsas_amd._capi import Context

pytestmark = pytest.mark.gpu

K, G = 8.3e5, 3.8e5


# stress and strain together: 8,382,528 bytes (below 8 MiB), 8,781,696 (five chunks),
# 25,632,288 (more chunks than the ring has slots, the last one partial)
@pytest.mark.parametrize("shape", [(21, 21, 22), (22, 21, 22), (33, 31, 29)])
def test_element_results_in_place(shape):
    print(f"[gpu] element results {shape}", flush=True)
    nx, ny, nz = shape
    sm = meshes.cube(nx, ny=ny, nz=nz, jitter=0.05, seed=6)
    c = Context(_capi.PRECISION_MIXED)
    try:
        c.set_nodes(sm.coords)
        c.add_tet_group(sm.tets, _capi.MAT_NEOHOOKEAN, (K, G))
        c.set_fixed_dofs(np.arange(3))
        c.finalize()
        U = 0.05 * np.sin(3 * sm.coords + np.array([0.1, 0.7, 1.9]))
        c.set_U(U.reshape(-1))
        x, u = sm.coords[sm.tets], U[sm.tets]
        F = np.eye(3) + (np.linalg.inv(x[:, 1:] - x[:, :1]) @ (u[:, 1:] - u[:, :1])).transpose(0, 2, 1)
        C = F.transpose(0, 2, 1) @ F
        Ci, J = np.linalg.inv(C), np.linalg.det(F)[:, None, None]
        P = F @ (G * (np.eye(3) - Ci) + K * J * (J - 1) * Ci)
        for _ in range(2):  # the ring is reused
            s, e = c.stress_strain(0, at_last_assembly=False)
            # FP64 on both sides, over some ten operations a value
            assert np.abs(e - C).max() <= 1e-12 * np.abs(C).max()
            assert np.abs(s - P).max() <= 1e-11 * np.abs(P).max()
    finally:
        c.close()
