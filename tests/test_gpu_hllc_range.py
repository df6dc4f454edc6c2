"""Right-hand sides whose HLLC operands approach the ends of the exponent range,
against the oracle (IEEE operations): velocities whose squares are subnormal, a
gas whose density products underflow, and speeds whose fourth powers overflow.
Bound as in test_gpu_parity, per variable: within 1e-12 of the largest flux over
the cell size (the flux scales of mass, momentum and energy below)."""
import numpy as np
import pytest

from helpers import config, init_text, oracle_for

pytestmark = pytest.mark.gpu

# density, pressure and velocity scales.  "slow": |v| from 1e-163 to 1e-160,
# a^2 = 0.14; "thin": density products 1e-310; "fast": |v|^2 a^2 = 1e312
CASES = {"slow": (1.0, 0.1, 1e-160), "thin": (1e-155, 1e-155, 0.3), "fast": (1.0, 1e156, 1e78)}


def _state(shape, case, gamma):
    rho0, p0, v0 = CASES[case]
    nz, ny, nx = shape
    z, y, x = np.meshgrid(*[(np.arange(m) + 0.5) / m for m in shape], indexing="ij")
    w = [2.0 * np.pi * a for a in (x, y, z)]
    rho = rho0 * (1.0 + 0.2 * np.sin(w[0]) + 0.1 * np.cos(w[1]))
    p = p0 * (1.0 + 0.1 * np.cos(w[0] + w[1]))
    if case == "slow":
        p = np.full(shape, p0)  # a contact: nothing but the velocities' tail moves
        f = v0 * np.exp(-7.0 * x)
    else:
        f = v0
    vel = [f * np.sin(w[0] + w[1]), f * np.cos(w[0] - w[1]), (f * np.sin(w[1] + w[2])) if nz > 1 else 0.0 * x]
    U = np.zeros((5,) + shape)
    U[0] = rho
    for a in range(3):
        U[1 + a] = rho * vel[a]
    U[4] = p / (gamma - 1.0) + 0.5 * rho * (vel[0] ** 2 + vel[1] ** 2 + vel[2] ** 2)
    return U


@pytest.mark.parametrize("dim,nq", [(2, 2), (2, 3), (3, 2), (3, 3)])
@pytest.mark.parametrize("case", sorted(CASES))
def test_operands_at_the_ends_of_the_exponent_range(case, dim, nq):
    import kfvm_amd
    n = (21, 18, 1) if dim == 2 else (18, 9, 6)
    # the indicator's threshold keeps every cell linear: the WENO weights take
    # fourth powers of the states, which do not reach as far
    c = config(dim=dim, n=n, nq=nq, bc="periodic", riemann="hllc", wenothresh="1.e30", fixeddt=1e-3,
               problem="quadrant2d" if dim == 2 else "riemann3d_planar", user=() if dim == 2 else (1.2,))
    text = init_text(c)
    s = kfvm_amd.Solver(init_text=text)
    f, d = s.weights
    o = oracle_for(c, kfvm_amd.parse_init(text), f, d)
    U = _state(s.shape[1:], case, c["gamma"])
    fl = np.zeros((2,) + s.shape[1:])
    fl[1] = 1.0
    for q in (s, o):
        q.state = U
        q.flags = fl
    s.eval_rhs()
    o.prime()
    K, R = s.rhs, o.rhs
    assert np.isfinite(R).all()
    assert np.isfinite(K).all()
    rho0, p0, v0 = CASES[case]
    speed, mom = v0 + np.sqrt(c["gamma"] * p0 / rho0), p0 + rho0 * v0 * v0
    scale = np.array([rho0 * speed, mom, mom, mom, mom * speed]) * max(n)
    worst = (np.abs(K - R).max(axis=(1, 2, 3)) / scale).max()
    print(f"[hllc] {case} {dim}D nq {nq}: max diff over the flux scale {worst:.3e}", flush=True)
    assert worst <= 1e-12
