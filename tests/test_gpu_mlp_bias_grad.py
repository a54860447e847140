"""Column sums of the guess network's bias gradient, 16 columns and 16 row
lanes a block: rows and columns below, at and above the 16 of a block."""
import numpy as np
import pytest

import polymer_amd as pa
from polymer_amd import geometry, guess

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 1), (15, 17), (16, 16), (17, 15), (128, 33), (1025, 225)])
def test_bias_gradient_is_the_column_sum(rows, cols):
    """One linear layer: db = sum_r 2 w (y - t) / sum w, with the device's own
    y.  Tolerance: each term is rounded at most four times and a column's sum
    has at most rows additions, (rows + 4) 2^-24 times the sum of |terms|."""
    print(f"case: bias gradient {rows} x {cols}", flush=True)
    ctx = pa.Context(pa.read_basis("STO-3G", geometry.water()))
    net = guess.MLP([8, cols], seed=5)
    rng = np.random.default_rng(11)
    x = rng.standard_normal((rows, 8)).astype(np.float32)
    t = rng.standard_normal((rows, cols)).astype(np.float32)
    w = rng.uniform(0.5, 1.0, (rows, cols)).astype(np.float32)
    y = guess.mlp_forward(net, ctx, x)
    guess.mlp_train_step(net, ctx, x, t, w, lr=0.0, update=False)
    dz = 2.0 * w.astype(np.float64) * (y.astype(np.float64) - t) / w.astype(np.float64).sum()
    db = net.grads()[-cols:]
    # y - t may cancel: its rounding is relative to |y| + |t|
    scale = (2.0 * w * (np.abs(y) + np.abs(t)) / w.sum()).sum(axis=0)
    assert np.all(np.abs(db - dz.sum(axis=0)) <= (rows + 4) * 2.0 ** -24 * scale)
    assert np.max(np.abs(db)) > 0
