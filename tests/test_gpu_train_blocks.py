"""Gradient sums of the indicator around their blocks: batches around 64 samples (one
workgroup) and around 32 workgroups (partials that are added in one go), against
the float64 gradient.  Bounds as in test_gpu_indicator: 1e-5 of the norm, for
sums of up to 2200 FP32 terms (random rounding: 2200^0.5 x 6e-8 = 3e-6)."""
import numpy as np
import pytest

import indicator_ref as ir

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 2047, 2048, 2049, 2200])
def test_gradient(dim, n):
    import kfvm_amd
    ind = kfvm_amd.Indicator(dim)
    rng = np.random.default_rng(n)
    nin, npar = ir.net_sizes(dim)
    P = rng.normal(0.0, 0.3, npar).astype(np.float32)
    X = rng.uniform(-1, 1, (n, nin)).astype(np.float32)
    Y = (rng.uniform(size=n) < 0.25).astype(np.float32)
    g, loss = ind.gradient(P, X, Y, pos_weight=4.0)
    lr, gr = ir.loss_and_grad(P, X, Y, dim, pos_weight=4.0)
    assert abs(loss - lr) <= 1e-5 * max(lr, 1e-3)
    assert np.linalg.norm(g - gr) <= 1e-5 * np.linalg.norm(gr)
