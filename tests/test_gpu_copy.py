"""States of several chunk sizes come back from the device as they went in: below
the size from which worker threads share the copy, just above it, and with a
last chunk that is not whole; from two threads at once too."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from helpers import config, init_text

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(64, 64), (640, 640), (701, 613), (1031, 811)])
def test_state_round_trip(n):
    import kfvm_amd
    s = kfvm_amd.Solver(init_text=init_text(config(dim=2, n=n + (1,), problem="quadrant2d", user=(), bc="outflow")))
    rng = np.random.default_rng(5)
    x = 1.0 + rng.random(s.shape)
    s.state = x
    assert np.array_equal(s.state, x)
    with ThreadPoolExecutor(2) as ex:
        for y in ex.map(lambda _: s.state, range(4)):
            assert np.array_equal(y, x)
    fl = rng.integers(0, 2, (2,) + s.shape[1:]).astype(float)
    s.flags = fl
    assert np.array_equal(s.flags, fl)
