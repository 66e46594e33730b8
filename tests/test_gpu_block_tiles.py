"""Jacobian blocks from one launch over all coloured directions, on grids at the
edges of 31 x 7 and 31 x 15 tiles: the exact blocks through J^T psi
(dot products with the oracle's J.v), the first-order ones (3 x 3 colours) through
the chunked ILU built from them, on the 3x3-box pattern and on the 13-point one,
where the slots that no direction writes have to be zero."""
import copy

import numpy as np
import pytest

import oracle_ffi as of
import precond_model as pm
from structured_amd import cases, lib

pytestmark = pytest.mark.gpu
SIZES = [(31, 14), (31, 15), (32, 16), (62, 21), (62, 30), (63, 31)]


def make(cols, rows, sa):
    case = cases.sa_bump(cols + 1, rows + 1, dy1=1e-3) if sa else cases.laminar_plate(cols + 1, rows + 1, dy1=5e-3)
    return case, case.perturbed_state(seed=5, amp=0.01)


@pytest.mark.parametrize("cols,rows", SIZES)
@pytest.mark.parametrize("sa", [False, True])
def test_exact_blocks(cols, rows, sa):
    case, q = make(cols, rows, sa)
    eq = lib.Equation(case)
    wd = eq.walldist() if sa else None
    rng = np.random.default_rng(cols + rows)
    psi = rng.standard_normal(q.shape)
    jt, _ = eq.jtv(q, psi)
    for _ in range(4):
        v = rng.standard_normal(q.shape)
        _, jv = of.jv(case, q, v, wd=wd)
        # J.v of the oracle and the library agree to 1e-10
        assert abs(np.vdot(psi, jv) - np.vdot(jt, v)) <= 1e-10 * np.abs(psi * jv).sum()
    eq.close()


@pytest.mark.parametrize("cols,rows", SIZES)
@pytest.mark.parametrize("sa", [False, True])
@pytest.mark.parametrize("precond", [6, 7])
def test_first_order_blocks(cols, rows, sa, precond):
    case, q = make(cols, rows, sa)
    eq = lib.Equation(case)
    wd = eq.walldist() if sa else None
    dt = eq.calc_dt(q, 50.0)
    eq.ls_preallocate(restart=4, precond=precond, maxit=4, rtol=1e-6)
    # leaves exact blocks, with all 13 slots, where the first-order ones go
    eq.ls_set_pc(2, 1.0, 32)
    eq.ls_set_lhs(q, dt)
    eq.ls_set_pc(1, 1.0, 32)
    eq.ls_set_lhs(q, dt)
    cj = copy.deepcopy(case)
    cj.order = 1
    nic, njc, nv = q.shape
    B = np.zeros((nic, njc, len(pm.SLOTS), nv, nv))
    I, Jx = np.meshgrid(np.arange(nic), np.arange(njc), indexing="ij")
    for a in range(5):
        for b in range(5):
            on = (I % 5 == a) & (Jx % 5 == b)
            for m in range(nv):
                e = np.zeros_like(q)
                e[..., m] = on
                _, jv = of.jv(cj, q, e, wd=wd)
                for s, (di, dj) in enumerate(pm.SLOTS):
                    ii, jj = I + di, Jx + dj
                    ok = (ii >= 0) & (ii < nic) & (jj >= 0) & (jj < njc) & (ii % 5 == a) & (jj % 5 == b)
                    B[:, :, s, :, m][ok] = jv[ok]
    v = np.random.default_rng(3).standard_normal(q.shape)
    z = eq.ls_precond_apply(v)
    zr = pm.ilu_chunked(B, 1.0 / dt[..., 0], v, 32, nine_point=precond == 7)
    err = float(np.abs(z - zr).max() / np.abs(zr).max())
    print(cols, rows, "sa", sa, "precond", precond, "err", err)
    # factors rounded to float32 on both sides: now and then one lands on the
    # other neighbour, 6e-8 away; a wrong block is off by more than 1e-3
    assert err <= 1e-6
    eq.close()
