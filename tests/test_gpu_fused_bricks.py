"""The fused sparse-mode path (k_linear_par, k_pp_rows, k_flux_par) against the
oracle on grids around its bricks (16 x 4 x 4, 2D 16 x 16): whole bricks, one
cell more and less, the smallest grids, every boundary condition and solver;
and weight tables without the mirror symmetry, which take the dense kernels.
Bounds as in test_gpu_parity: first RHS within 1e-12 of the largest RHS, equal
WENO flags, one fixed-dt step within 1e-12 per cell."""
import numpy as np
import pytest

from helpers import cell_rel_diff, config, init_text, oracle_for

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _check(c, weights=None):
    import kfvm_amd
    text = init_text(c)
    s = kfvm_amd.Solver(init_text=text)
    p = kfvm_amd.parse_init(text)
    f, d = s.weights
    if weights is not None:
        f, d = weights(f), d
        s.set_weights(f, d)
    o = oracle_for(c, p, f, d)
    o.set_ic(c["problem"], p["user"], p["seed"])
    fl = np.zeros((2,) + s.shape[1:])
    fl[1] = 1.0
    s.flags = fl
    o.flags = fl
    s.eval_rhs()
    o.prime()
    K, R = s.rhs, o.rhs
    rk = np.abs(K - R).max() / max(np.abs(R).max(), 1e-300)
    assert rk <= TOL
    assert np.array_equal(s.flags[0], o.flags[0])
    assert s.take_step() == o.take_step() == 0
    r = cell_rel_diff(s.state, o.state).max()
    print(f"[bricks] {c['n']} {c['bc']} {c['riemann']}: RHS {rk:.2e}, step {r:.2e}", flush=True)
    assert r <= TOL


@pytest.mark.parametrize("n,bc,riemann", [
    ((16, 4, 4), "outflow", "hllc"), ((17, 5, 5), "periodic", "hllc"), ((15, 3, 7), "reflecting", "hll"),
    ((33, 9, 2), "noslip", "llf"), ((2, 2, 2), "periodic", "hllc"), ((31, 8, 11), "outflow", "hllc"),
])
def test_bricks_3d(n, bc, riemann):
    _check(config(n=n, bc=bc, riemann=riemann, user=(1.2,), fixeddt=0.002))


@pytest.mark.parametrize("nq", [2, 3])
@pytest.mark.parametrize("n,bc,riemann", [
    ((16, 16), "outflow", "hllc"), ((17, 15), "periodic", "hll"), ((2, 33), "reflecting", "hllc"),
    ((49, 31), "noslip", "llf"),
])
def test_bricks_2d(n, bc, riemann, nq):
    _check(config(dim=2, n=n + (1,), nq=nq, bc=bc, riemann=riemann, problem="quadrant2d", seed=9, user=(),
                  fixeddt=0.001))


@pytest.mark.parametrize("dim", [2, 3])
def test_tables_without_the_symmetry_take_the_dense_kernels(dim):
    def skew(f):
        g = f.copy()
        g[0, 0, 0, :2] += np.array([1e-6, -1e-6])  # keeps the sum of the row
        return g

    if dim == 3:
        _check(config(n=(18, 6, 5), fixeddt=0.002), skew)
    else:
        _check(config(dim=2, n=(20, 18, 1), problem="quadrant2d", seed=3, user=(), fixeddt=0.001), skew)
