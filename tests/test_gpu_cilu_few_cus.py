"""The chunked line ILU as on a device on which not every CU takes part (one lane a
row, a launch per pass) against the same factors with both passes in one launch:
chunk widths, four and five unknowns, both patterns and directions, partial last
chunks and more rows than the ring of solved steps holds."""
import ctypes as C

import numpy as np
import pytest

from structured_amd import cases, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols,rows,sa", [(77, 70, True), (33, 3, True), (70, 67, False), (49, 8, False)])
@pytest.mark.parametrize("width", [8, 16, 24, 32])
@pytest.mark.parametrize("precond", [6, 7])
def test_a_launch_per_pass(cols, rows, sa, width, precond):
    case = cases.sa_bump(cols + 1, rows + 1, dy1=1e-3) if sa else cases.laminar_plate(cols + 1, rows + 1, dy1=5e-3)
    q = case.perturbed_state(seed=6, amp=0.01)
    eq = lib.Equation(case)
    dt = eq.calc_dt(q, 50.0)
    v = [np.random.default_rng(s).standard_normal(q.shape) for s in (1, 2)]
    z = []
    for few in (0, 1):
        assert lib.load().sg_test_few_cus(eq.h, C.c_int(few)) == 1 - few
        eq.ls_preallocate(restart=4, precond=precond, maxit=4, rtol=1e-6)
        eq.ls_set_pc(1 if precond == 7 else 0, 1.0, width)
        eq.ls_set_lhs(q, dt)
        z.append([eq.ls_precond_apply(x, transpose=t) for t in (False, True) for x in v])
    for a, b in zip(*z):
        err = float(np.abs(a - b).max() / np.abs(a).max())
        print(cols, rows, "sa", sa, "width", width, "precond", precond, "err", err)
        # the same float32 factors; the FP64 sums of a row in another order
        assert err <= 1e-10
    eq.close()
