"""Cleaning speed c_h of GLM-MHD flows whose internal energy is a small part of
the total: the right-hand side of psi, -c_h^2 div B at psi = 0, against the
oracle.  In a weakly magnetised flow of Mach number 134 (E = 1e4 e) c_h is the
sound speed of the face states, so a relative error in their internal energy
appears in psi's right-hand side.  Rounding: a face state's dot product is good
to about three units of E (3 x 1.1e-16 x 1e4 = 3e-12 of e each side, 1.4e-11
with the largest of many points taken on both); an offset of 1e-14 E would show
as 1e-10.  Bound: 3e-11 of the largest value."""
import numpy as np
import pytest

from helpers import config, init_text, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,nq", [(2, 2), (2, 3), (3, 2), (3, 3)])
def test_cleaning_speed_of_a_cold_flow(dim, nq):
    import kfvm_amd
    n = (18, 17, 1) if dim == 2 else (17, 9, 6)
    c = config(dim=dim, n=n, nq=nq, equation="mhd_glm", riemann="llf", bc="periodic", gamma=5.0 / 3.0, user=(),
               problem="orszag_tang" if dim == 2 else "mhd_vortex3d", wenothresh="1.e30", fixeddt=1e-4)
    text = init_text(c)
    s = kfvm_amd.Solver(init_text=text)
    f, d = s.weights
    o = oracle_for(c, kfvm_amd.parse_init(text), f, d)
    shape = s.shape[1:]
    z, y, x = np.meshgrid(*[(np.arange(m) + 0.5) / m for m in shape], indexing="ij")
    U = np.zeros((9,) + shape)
    U[0] = 1.0
    U[1], U[2] = np.sqrt(2e4), 1e-3 * np.sin(2.0 * np.pi * x)
    U[5] = 1e-3 * np.sin(2.0 * np.pi * x)  # div B: what psi's right-hand side measures c_h by
    U[6] = 1e-3 * np.cos(2.0 * np.pi * x)
    U[4] = 1.0 + 0.5 * (U[1] ** 2 + U[2] ** 2 + U[5] ** 2 + U[6] ** 2)
    fl = np.zeros((2,) + shape)
    fl[1] = 1.0
    for q in (s, o):
        q.state = U
        q.flags = fl
    s.eval_rhs()
    o.prime()
    assert not s.flags[0].any() and (s.flags[1] == 1.0).all()
    K, R = s.rhs[8], o.rhs[8]
    r = np.abs(K - R).max() / np.abs(R).max()
    print(f"[mhd] cleaning speed, {dim}D nq {nq}: psi's right-hand side {r:.3e} off", flush=True)
    assert r <= 3e-11
