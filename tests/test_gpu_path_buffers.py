"""Device memory of the two sparse-mode paths: a 3D Euler solver that takes the
learned selection gives the fused path's surface planes back and gets them again
without it, and evaluates as a solver that never switched."""
import ctypes

import numpy as np
import pytest

from helpers import config, init_text

pytestmark = pytest.mark.gpu


def test_selection_keeps_one_path_s_buffers():
    import kfvm_amd
    from kfvm_amd import train_indicator
    kfvm_amd.load_library()
    hip = ctypes.CDLL("libamdhip64.so.7")  # the library's own HIP runtime

    def free():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipDeviceSynchronize() == 0
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    n = (96, 80, 72)
    cells = n[0] * n[1] * n[2]
    c = config(n=n, fixeddt=0.001)
    s = kfvm_amd.Solver(init_text=init_text(c))
    ref = kfvm_amd.Solver(init_text=init_text(c))
    for q in (s, ref):
        q.eval_rhs()  # what the first evaluation allocates by itself
    start = free()
    s.set_indicator(train_indicator.load("euler3d"), 0.0)
    on = start - free()
    # the compact WENO staging (a row of 120 for every fourth cell) and the
    # admissibility flags come, the surface planes (2 (n / B + 1) planes of 20
    # values an axis, B = 16, 4, 4) go; 4 MB for the allocator's granularity
    staging = cells // 4 * 120 * 8
    planes = sum(2 * (-(-n[a] // b) + 1) * 20 * (cells // n[a]) for a, b in ((0, 16), (1, 4), (2, 4))) * 8
    print(f"[memory] learned selection on: {on / 1e6:.1f} MB, staging {staging / 1e6:.1f}, planes {planes / 1e6:.1f}",
          flush=True)
    assert planes > 50e6
    assert on <= staging + 8 * cells - planes + 4 * 2**20
    s.set_indicator(None)
    off = start - free()
    print(f"[memory] off again: {off / 1e6:.1f} MB", flush=True)
    assert off <= 8 * cells + 4 * 2**20
    for q in (s, ref):
        q.eval_rhs()
        assert q.take_step() == 0
    assert np.array_equal(s.state, ref.state)
