"""Arnoldi steps at the edges of the fused reductions: basis sizes on both
sides of a group of eight vectors, restarts of one vector, grids whose vectors
fill less than one block up to several slices, four and five unknowns, and
the transposed operator.  The residual that FGMRES reports comes from its
rotations; the true one is formed from the oracle's J.v."""
import numpy as np
import pytest

import oracle_ffi as of
from structured_amd import cases, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj,sa", [(4, 4, False), (33, 9, True), (70, 37, False), (65, 49, True)])
@pytest.mark.parametrize("restart,maxit", [(1, 5), (7, 14), (8, 8), (9, 20), (33, 40)])
def test_reported_residual_is_the_true_one(ni, nj, sa, restart, maxit):
    case = cases.sa_bump(ni, nj, dy1=1e-3) if sa else cases.laminar_plate(ni, nj, dy1=1e-2)
    q = case.perturbed_state(seed=4, amp=0.002)
    eq = lib.Equation(case)
    dt = eq.calc_dt(q, 5.0)
    r, _ = eq.calc_residual(q)
    eq.ls_preallocate(restart=restart, precond=0, maxit=maxit, rtol=1e-13)
    eq.ls_set_lhs(q, dt)
    eq.ls_set_rhs(r)
    dq, it, rr = eq.ls_solve()
    _, jdq = of.jv(case, q, dq, wd=eq.walldist() if sa else None)
    true = np.linalg.norm(dq / dt - jdq - r) / np.linalg.norm(r)
    print(ni, nj, sa, restart, "iters", it, "relres", rr, "true", true)
    # as in the linear-solve test: the rotations' estimate against the true
    # residual, which carries the rounding of J.v (1e-10)
    assert abs(true - rr) <= 1e-3 * rr + 1e-10
    assert np.isfinite(dq).all()
    # the same solve again: nothing is left over in the reductions
    dq2, it2, rr2 = eq.ls_solve()
    assert it2 == it and rr2 == rr and np.array_equal(dq, dq2)
    eq.close()
