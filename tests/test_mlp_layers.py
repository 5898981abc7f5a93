"""The perceptron's tiled layer and gradient kernels against a float64
restatement, at sizes around their tiles of 64 and their chunks of 32 rows.

Tolerances: an output is a sum of at most max(n, 200) products in FP32, in
chains of at most 256 and chunk sums behind them; each rounding is 2^-24 of a
partial sum, so the error of a gradient is below 600 * 2^-24 = 3.6e-5 of the
sum of its terms' magnitudes.  Three layers in a row at most triple it: 1.1e-4
of the largest gradient's magnitudes (whose terms these bound), 2e-4 used."""
import numpy as np
import pytest

import mlp_oracle as mo
import tagmatch_amd as tm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,n", [((16, 64, 3), 1), ((16, 64, 3), 33), ((16, 64, 3), 8193), ((1, 65, 1), 64),
                                     ((200, 63, 70), 65), ((3, 130, 129), 31)])
def test_gradients_vs_float64(gpu, shape, n):
    m = tm.MLP(*shape, seed=5)
    rng = np.random.default_rng(n)
    x = rng.normal(0, 1, (n, shape[0])).astype(np.float32)
    t = rng.normal(0, 1, (n, shape[2])).astype(np.float32)
    loss, g = m.loss_grad(x, t)
    le, ge = mo.loss_grad(m.params(), x, t, shape)
    ga = mo.loss_grad(np.abs(m.params()), np.abs(x), -np.abs(t), shape)[1]   # magnitudes of the terms
    assert loss == pytest.approx(le, rel=1e-5)
    assert np.all(np.abs(g - ge) <= 2e-4 * np.maximum(np.abs(ga), np.abs(ge)) + 1e-7)
