"""The KXRCF selector appends one block of cells at a time to the WENO list: grids
around its block sizes (1024 cells; 512 with the 3D 3x3 rule), against the oracle.
The flags are equal and the first RHS within 1e-12 of the largest RHS."""
import numpy as np
import pytest

from helpers import config, init_text, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,nq,n", [
    (2, 2, (31, 33, 1)), (2, 2, (32, 32, 1)), (2, 2, (41, 25, 1)), (2, 3, (41, 50, 1)),
    (3, 2, (11, 13, 7)), (3, 3, (7, 37, 2)), (3, 3, (8, 8, 8)), (3, 3, (9, 19, 3)),
])
def test_selected_cells_and_rhs(dim, nq, n):
    import kfvm_amd
    c = config(dim=dim, n=n, nq=nq, bc="outflow", **({"problem": "quadrant2d", "user": ()} if dim == 2 else {}))
    text = init_text(c)
    s = kfvm_amd.Solver(init_text=text)
    p = kfvm_amd.parse_init(text)
    f, d = s.weights
    o = oracle_for(c, p, f, d)
    o.set_ic(c["problem"], p["user"], p["seed"])
    fl = np.zeros((2,) + s.shape[1:])
    fl[1] = 1.0
    s.flags = fl
    o.flags = fl
    s.eval_rhs()
    o.prime()
    rk = np.abs(s.rhs - o.rhs).max() / max(np.abs(o.rhs).max(), 1e-300)
    print(f"[select] {n} nq {nq}: RHS {rk:.2e}, WENO cells {int(s.flags[0].sum())}", flush=True)
    assert np.array_equal(s.flags[0], o.flags[0])
    assert rk <= 1e-12
