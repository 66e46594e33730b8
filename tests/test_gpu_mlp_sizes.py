"""The fused network kernel at the edges of its tiles: a wave's 32 rows, a
block's 128, and the row counts past which waves take several tiles.  Against
the numpy model with the kernel's BF16 rounding points; tolerances as for the
gradients at the ordinary sizes (a BF16 rounding that falls on the other side
moves one row's contribution by 2^-9)."""
import numpy as np
import pytest

import mlp_model as mm
from structured_amd import lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 33, 129, 32768, 32769, 70001])
def test_loss_gradient_forward_sizes(n):
    rng = np.random.default_rng(n)
    net = lib.Mlp(max_rows=n, seed=3)
    p = (mm.glorot(seed=2) + 0.02 * rng.standard_normal(mm.NPARAM)).astype(np.float32)
    net.params = p
    x = rng.uniform(-1.0, 1.0, (n, 5)).astype(np.float32)
    t = (0.3 * np.tanh(1.5 * x[:, 0] - x[:, 2] + 0.5 * x[:, 3] * x[:, 4]) + 0.05).astype(np.float32)
    loss, g = net.loss_grad(x, t)
    lm, gm = mm.loss_grad(p.astype(np.float64), x, t, bf=True)
    # one row alone: its loss can be small against the rounding of y (2e-4 at a flip)
    assert abs(loss - lm) <= (1e-4 * lm if n > 100 else 1e-4 * lm + 4e-4 * np.sqrt(lm))
    for k, (o, shp) in mm.OFF.items():
        cnt = int(np.prod(shp)) if shp else 1
        rel = np.linalg.norm(g[o:o + cnt] - gm[o:o + cnt]) / max(np.linalg.norm(gm[o:o + cnt]), 1e-30)
        print(n, "grad %s rel %.2e" % (k, rel))
        assert rel <= (2e-3 if n > 100 else 1e-2), k
    y = net.forward(x)
    ym, _ = mm.forward(p.astype(np.float64), x, bf=True)
    assert np.median(np.abs(y - ym)) <= 2e-6 + (n < 100) * 1e-3 and np.abs(y - ym).max() <= 1e-3
