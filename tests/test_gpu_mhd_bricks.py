"""The GLM-MHD linear pass in mirror-symmetric form (k_mhd_linear_par) against the
oracle on grids around its bricks (16 x 8 x 4, 2D 16 x 16), every boundary
condition, and weight tables without the symmetry, which take the dense kernel.
Bounds as in test_gpu_parity: first RHS within 1e-12 of the largest RHS, equal
WENO flags, one fixed-dt step within 1e-12 per cell."""
import numpy as np
import pytest

from test_gpu_fused_bricks import _check
from helpers import config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bc,riemann,nq", [
    ((16, 8, 4), "periodic", "llf", 2), ((17, 9, 5), "outflow", "hll", 2), ((15, 7, 3), "reflecting", "kepes", 2),
    ((2, 2, 2), "periodic", "llf", 2), ((9, 10, 6), "periodic", "llf", 3),
])
def test_mhd_bricks_3d(n, bc, riemann, nq):
    _check(config(n=n, nq=nq, equation="mhd_glm", riemann=riemann, problem="mhd_blast", user=(0.2, 0.5, 0.0), bc=bc,
                  gamma=5.0 / 3.0, fixeddt=0.0005))


@pytest.mark.parametrize("nq", [2, 3])
@pytest.mark.parametrize("n,bc,riemann", [
    ((16, 16), "periodic", "kepes"), ((17, 15), "outflow", "hll"), ((31, 33), "reflecting", "llf"),
])
def test_mhd_bricks_2d(n, bc, riemann, nq):
    _check(config(dim=2, n=n + (1,), nq=nq, equation="mhd_glm", riemann=riemann, problem="orszag_tang", user=(),
                  bc=bc, gamma=5.0 / 3.0, fixeddt=0.0005))


@pytest.mark.parametrize("dim", [2, 3])
def test_mhd_tables_without_the_symmetry(dim):
    def skew(f):
        g = f.copy()
        g[0, 0, 0, :2] += np.array([1e-6, -1e-6])  # keeps the sum of the row
        return g

    n = (18, 9, 5) if dim == 3 else (18, 17, 1)
    _check(config(dim=dim, n=n, equation="mhd_glm", riemann="llf", problem="mhd_blast", user=(0.2, 0.5, 0.0),
                  bc="outflow", gamma=5.0 / 3.0, fixeddt=0.0005), skew)
