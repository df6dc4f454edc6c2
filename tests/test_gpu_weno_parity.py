"""KFVM-WENO in mirror-symmetric form (k_weno_par) against the oracle: cell counts
around its blocks of 64, walls that negate variables, anisotropic cells, with a
list (KXRCF) and on every cell (negative threshold), and derivative tables without
the symmetry, which take the dense kernels.  Bounds as in test_gpu_parity."""
import numpy as np
import pytest

from helpers import config
from test_gpu_fused_bricks import _check

pytestmark = pytest.mark.gpu

HYDRO2 = dict(dim=2, problem="quadrant2d", seed=9, user=(), fixeddt=0.001)
MHD = dict(equation="mhd_glm", problem="mhd_blast", user=(0.2, 0.5, 0.0), gamma=5.0 / 3.0, fixeddt=0.0005)


@pytest.mark.parametrize("nq", [2, 3])
@pytest.mark.parametrize("n,bc,thresh", [
    ((9, 7), "outflow", -1.0), ((8, 8), "reflecting", -1.0), ((13, 5), "noslip", -1.0), ((2, 2), "periodic", -1.0),
    ((37, 29), "reflecting", 1.0), ((43, 3), "noslip", 1.0),
])
def test_euler_2d(n, bc, thresh, nq):
    _check(config(n=n + (1,), nq=nq, bc=bc, riemann="hllc", wenothresh=thresh, hi=(1.0, 0.4, 1.0), **HYDRO2))


@pytest.mark.parametrize("n,bc,nq", [
    ((13, 10, 7), "reflecting", 2), ((9, 21, 4), "noslip", 2), ((2, 3, 50), "outflow", 2), ((10, 9, 8), "reflecting", 3),
    ((6, 5, 4), "periodic", 3),
])
def test_euler_3d_listed(n, bc, nq):
    _check(config(n=n, nq=nq, bc=bc, riemann="hllc", user=(1.2,), fixeddt=0.001, hi=(1.0, 0.7, 1.3)))


@pytest.mark.parametrize("n,bc,nq,thresh", [
    ((9, 7, 1), "outflow", 2, -1.0), ((13, 5, 1), "reflecting", 3, -1.0), ((21, 23, 1), "reflecting", 2, 1.0),
    ((7, 3, 3), "outflow", 2, -1.0), ((4, 4, 4), "reflecting", 2, -1.0), ((5, 4, 3), "periodic", 3, -1.0),
    ((9, 10, 6), "reflecting", 2, 1.0),
])
def test_mhd(n, bc, nq, thresh):
    _check(config(dim=3 if n[2] > 1 else 2, n=n, nq=nq, bc=bc, riemann="llf", wenothresh=thresh, **MHD))


@pytest.mark.parametrize("dim", [2, 3])
def test_derivatives_without_the_symmetry(dim):
    import kfvm_amd
    from helpers import init_text

    c = config(n=(9, 8, 1), bc="outflow", riemann="hllc", wenothresh=-1.0, **HYDRO2) if dim == 2 else \
        config(n=(8, 7, 5), bc="outflow", riemann="hllc", user=(1.2,), fixeddt=0.001)
    a, b = kfvm_amd.Solver(init_text=init_text(c)), kfvm_amd.Solver(init_text=init_text(c))
    f, d = a.weights
    d = d.copy()
    d[0, 0, 1] += 1e-9
    a.set_weights(f, d)
    a.eval_rhs()
    b.eval_rhs()
    # the changed row alters the smoothness indicators by 1e-9 of their size
    assert 0.0 < np.abs(a.rhs - b.rhs).max() <= 1e-6 * np.abs(b.rhs).max()
