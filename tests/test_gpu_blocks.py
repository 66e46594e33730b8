"""Jacobian blocks from one launch over all coloured directions, on grids at
the edges of the residual's 31 x 7 tiles: the exact blocks through J^T psi
(the dot-product identity with J.v, and the oracle's J.v on unit vectors)."""
import numpy as np
import pytest

import oracle_ffi as of
from structured_amd import cases, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols,rows", [(3, 3), (31, 7), (32, 8), (33, 15), (62, 6), (63, 21)])
@pytest.mark.parametrize("sa,flux", [(False, "roe"), (True, "roe"), (True, "ausm")])
def test_blocks_give_the_transposed_product(cols, rows, sa, flux):
    case = cases.sa_bump(cols + 1, rows + 1, dy1=1e-3) if sa else cases.laminar_plate(cols + 1, rows + 1, dy1=1e-2)
    case.flux = flux
    q = case.perturbed_state(seed=5, amp=0.01)
    eq = lib.Equation(case)
    rng = np.random.default_rng(cols + rows)
    v, psi = rng.standard_normal(q.shape), rng.standard_normal(q.shape)
    jt, _ = eq.jtv(q, psi)
    jv = eq.jv(q, v)
    a, b = np.vdot(psi, jv), np.vdot(jt, v)
    scale = np.abs(psi * jv).sum()
    print(cols, rows, sa, flux, a, b)
    assert abs(a - b) <= 1e-12 * scale
    # single entries: (J^T psi)_c = psi . J e_c with the oracle's J.v
    wd = eq.walldist() if sa else None
    for _ in range(3):
        c = (int(rng.integers(cols)), int(rng.integers(rows)), int(rng.integers(q.shape[2])))
        e = np.zeros_like(q)
        e[c] = 1.0
        _, je = of.jv(case, q, e, wd=wd)
        assert abs(jt[c] - np.vdot(psi, je)) <= 1e-10 * np.abs(psi * je).sum() + 1e-300
    eq.close()
