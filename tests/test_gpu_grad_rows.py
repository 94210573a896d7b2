"""One-off gradient of the cost model on both sides of the wide launch's
smallest row count, against an FP64 numpy gradient."""
import numpy as np
import pytest

from test_mlp import data, np_grad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 65, 255, 256, 257, 3073, 50021])
def test_gradient_rows(mce, rows):
    x, y = data(rows + 1, 7)
    m = mce.mlp_init(x, seed=9)
    x, y = x[:rows], y[:rows]
    P = {k: (v.astype(np.float64) if isinstance(v, np.ndarray) else v) for k, v in mce.mlp_params(m).items()}
    g, loss = mce.mlp_grad(m, x, y)
    g2, loss2 = mce.mlp_grad(m, x, y)
    assert np.array_equal(g, g2) and loss == loss2  # no sum depends on timing
    xd, yd = x.astype(np.float64), y.astype(np.float64)
    ref, ref_loss = np_grad(P, xd, yd)
    # a row's forward and backward pass in FP32 is good to some 200 roundings
    # (6e-8 each); a hidden unit within that of its kink may fall on the other
    # side in one row, which moves a component by that row's share
    share = 1e-5 + 4.0 / rows
    assert abs(loss - ref_loss) <= 2e-5 * max(1.0, ref_loss)
    assert np.abs(g - ref).max() <= (share if rows > 200 else 1e-4) * np.abs(ref).max()
