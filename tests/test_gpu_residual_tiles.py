"""The residual and J.v on grids at the edges of the tiles (31 columns by 7 or
15 rows of cells) and on grids whose rows of tiles take the taller ones,
against the oracle; the norms against the residual they belong to."""
import numpy as np
import pytest

import oracle_ffi as of
from structured_amd import cases, lib

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


# 7-row tiles up to 512 of them; 15-row tiles where they need fewer turns of
# the chip: 496 x 240 fills 16 x 16 of them, the others leave a ragged end
SIZES = [(3, 3), (30, 6), (31, 7), (32, 8), (33, 15), (62, 14), (63, 22), (496, 240), (495, 239), (466, 254), (3840, 29)]


@pytest.mark.parametrize("cols,rows", SIZES)
@pytest.mark.parametrize("sa,flux,order", [(False, "ausm", 2), (True, "roe", 2), (True, "roe", 1)])
def test_tiles_vs_oracle(cols, rows, sa, flux, order):
    case = cases.sa_bump(cols + 1, rows + 1, dy1=1e-3) if sa else cases.laminar_plate(cols + 1, rows + 1, dy1=1e-3)
    case.flux, case.order = flux, order
    q = case.perturbed_state(seed=7, amp=0.01)
    v = np.random.default_rng(cols).standard_normal(q.shape) * np.abs(q).max(axis=(0, 1))
    wd = of.wall_distance(case) if sa else None
    eq = lib.Equation(case)
    for _ in range(2):  # the second launch finds the slots as the first left them
        r, l2 = eq.calc_residual(q)
        ro, _ = of.residual(case, q, wd=wd)
        assert rel(r, ro) <= 1e-11
        np.testing.assert_allclose(l2, np.sqrt((r ** 2).sum(axis=(0, 1))), rtol=1e-12)
    assert rel(eq.jv(q, v), of.jv(case, q, v, wd=wd)[1]) <= 1e-10
    eq.close()


@pytest.mark.parametrize("cols,rows", [(3, 3), (31, 7), (32, 8), (495, 239)])
@pytest.mark.parametrize("sa", [False, True])
def test_stages_written_by_the_residual(cols, rows, sa):
    """A Runge-Kutta step, whose stages are the residual kernel's output,
    against its residuals and time steps taken one by one."""
    import torch
    case = cases.sa_bump(cols + 1, rows + 1, dy1=1e-3) if sa else cases.laminar_plate(cols + 1, rows + 1, dy1=1e-3)
    q0 = case.perturbed_state(seed=3, amp=0.01)
    eq = lib.Equation(case)
    dev = torch.device("cuda:0")
    aos = torch.from_numpy(np.ascontiguousarray(q0).reshape(-1)).to(dev)
    qd = torch.zeros(eq.nvar * eq.plane, dtype=torch.float64, device=dev)
    eq.aos_to_soa_dev(aos.data_ptr(), qd.data_ptr())
    eq.synchronize()
    l2 = eq.step_explicit_dev(qd.data_ptr(), "rk4_jameson", 0.5)
    eq.soa_to_aos_dev(qd.data_ptr(), aos.data_ptr())
    eq.synchronize()
    got = aos.cpu().numpy().reshape(q0.shape)
    dt, q = eq.calc_dt(q0, 0.5), q0
    for s in range(4):
        r, norms = eq.calc_residual(q)
        q = q0 + (r * dt) / (4.0 - s)
    # the same operations on the same residuals; the host's and the device's
    # square root and divisions may differ in the last place
    for m in range(eq.nvar):
        assert rel(got[..., m], q[..., m]) <= 1e-13
    np.testing.assert_allclose(l2, norms, rtol=1e-10)
    eq.close()
