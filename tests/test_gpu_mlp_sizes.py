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
    # a row's output does not depend on where in a tile or batch it lies
    y = net.forward(x)
    cut = n // 3
    assert np.array_equal(y, np.concatenate([net.forward(x[:cut]), net.forward(x[cut:])]))


def shuffle(n, epochs, seed):
    """The documented shuffle on the host: splitmix64 draws, Fisher-Yates."""
    s, mask, out = seed, (1 << 64) - 1, []
    for _ in range(epochs):
        p = np.arange(n)
        for k in range(n - 1, 0, -1):
            s = (s + 0x9E3779B97F4A7C15) & mask
            z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & mask
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
            j = (z ^ (z >> 31)) % (k + 1)
            p[k], p[j] = p[j], p[k]
        out.append(p)
    return out


@pytest.mark.parametrize("n,batch", [(1, 1), (2, 1), (3, 3), (257, 100), (5000, 700)])
def test_training_order_is_the_seeded_shuffle(n, batch):
    """Three epochs of minibatch steps equal the same steps taken one by one
    on the rows that the host's shuffle gives, bit for bit (the step counter
    of Adam runs on across the calls)."""
    rng = np.random.default_rng(n)
    x = rng.uniform(-1.0, 1.0, (n, 5)).astype(np.float32)
    t = rng.uniform(-0.3, 0.3, n).astype(np.float32)
    p = mm.glorot(seed=5).astype(np.float32)
    a, b = lib.Mlp(max_rows=batch, seed=1), lib.Mlp(max_rows=batch, seed=1)
    a.params, b.params = p, p
    hist = a.train(x, t, epochs=3, batch=batch, lr=1e-2, seed=9)
    for e, perm in enumerate(shuffle(n, 3, 9)):
        losses = []
        for k in range(n // batch):
            rows = perm[k * batch:(k + 1) * batch]
            # a full-batch step shuffles its rows again: undo that order first
            inv = np.empty(batch, dtype=np.int64)
            inv[shuffle(batch, 1, 4)[0]] = np.arange(batch)
            losses.append(b.train(x[rows][inv], t[rows][inv], epochs=1, batch=batch, lr=1e-2, seed=4)[0])
        assert abs(np.mean(np.float64(losses)) - hist[e]) <= 1e-7 * hist[e]
        # (float32 mean of the same losses)
    assert np.array_equal(a.params, b.params)
