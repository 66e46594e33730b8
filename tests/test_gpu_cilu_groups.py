"""The chunked line ILU's column groups at their edges: a last chunk of one
column, chunks that fill one group exactly or leave one column to the next,
more rows than the ring of solved steps holds, the fewest rows a grid can
have, both stencil patterns and both directions.  The reference is the numpy
model with float32 factors on Jacobian blocks from the oracle's coloured
J.v products."""
import copy

import numpy as np
import pytest

import oracle_ffi as of
import precond_model as pm
from structured_amd import cases, lib

pytestmark = pytest.mark.gpu


def oracle_blocks(case, q, wd):
    """Blocks of the 13-point stencil: 5 x 5 colours times nv products."""
    nic, njc, nv = q.shape
    B = np.zeros((nic, njc, len(pm.SLOTS), nv, nv))
    I, Jx = np.meshgrid(np.arange(nic), np.arange(njc), indexing="ij")
    for a in range(5):
        for b in range(5):
            on = (I % 5 == a) & (Jx % 5 == b)
            for m in range(nv):
                v = np.zeros_like(q)
                v[..., m] = on
                _, jv = of.jv(case, q, v, wd=wd)
                for s, (di, dj) in enumerate(pm.SLOTS):
                    ii, jj = I + di, Jx + dj
                    ok = (ii >= 0) & (ii < nic) & (jj >= 0) & (jj < njc) & (ii % 5 == a) & (jj % 5 == b)
                    B[:, :, s, :, m][ok] = jv[ok]
    return B


@pytest.mark.parametrize("cols,rows,sa,width", [
    (33, 3, True, 32),    # a chunk of one column, three rows
    (23, 131, True, 32),  # groups of 6, the last of 5; the ring wraps
    (11, 70, True, 32),   # a group of 6 and one of 5 of a chunk whose others are absent
    (24, 9, False, 24),   # three groups of 8
    (30, 67, False, 32),  # nv = 4, groups of 8, the last of 6; the ring wraps
    (17, 66, False, 16),  # nv = 4: two groups of 8, then one column
    (6, 65, True, 32),    # one group of 6, nv 5
    (13, 12, True, 16),
    (8, 64, False, 8),    # one group of 8, nv 4
    (25, 5, False, 32),
])
@pytest.mark.parametrize("precond", [6, 7])
def test_groups_match_model(cols, rows, sa, width, precond):
    ni, nj = cols + 1, rows + 1
    case = cases.sa_bump(ni, nj, dy1=1e-3) if sa else cases.laminar_plate(ni, nj, dy1=5e-3)
    q = case.perturbed_state(seed=6, amp=0.01)
    eq = lib.Equation(case)
    dt = eq.calc_dt(q, 50.0)
    nine = precond == 7
    eq.ls_preallocate(restart=10, precond=precond, maxit=10, rtol=1e-6)
    eq.ls_set_pc(1 if nine else 0, 1.0, width)
    eq.ls_set_lhs(q, dt)
    cj = copy.deepcopy(case)
    if nine:
        cj.order = 1
    B = oracle_blocks(cj, q, eq.walldist() if sa else None)
    rng = np.random.default_rng(3)
    for transpose in (False, True):
        v = rng.standard_normal(q.shape)
        eq.ls_precond_apply(rng.standard_normal(q.shape), transpose=transpose)  # leaves nothing for the next apply
        z = eq.ls_precond_apply(v, transpose=transpose)
        zr = pm.ilu_chunked(B, 1.0 / dt[..., 0], v, width, transpose=transpose, nine_point=nine)
        err = float(np.abs(z - zr).max() / np.abs(zr).max())
        print(cols, rows, "sa", sa, "width", width, "precond", precond, "transpose", transpose, "err", err)
        # the factors are rounded to float32 on both sides from FP64 values that
        # agree to about 1e-12: now and then one lands on the other neighbour,
        # 6e-8 away; a wrong row or column is off by more than 1e-3
        assert err <= 1e-6
    eq.close()
