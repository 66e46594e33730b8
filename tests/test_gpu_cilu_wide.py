"""The chunked line ILU on grids so wide that its apply takes one lane a row
(more than 256 column groups of the two-lane layout), and at the last width
below that: every chunk width, four and five unknowns, both stencil patterns
and both directions, last chunks of one column, of part of a group and of a
group and a bit, the fewest rows a grid can have and more rows than the ring of
solved steps holds.  Chunks do not couple, so the numpy model with float32
factors (on Jacobian blocks from the oracle's coloured J.v products) is formed
for some of them: the first, one inside, and the last two."""
import copy

import numpy as np
import pytest

import oracle_ffi as of
import precond_model as pm
from structured_amd import cases, lib

pytestmark = pytest.mark.gpu


def oracle_blocks(case, q, wd, per):
    """Blocks of the 13-point stencil (per 5) or the 3x3 box (per 3): per x per
    colours times nv products."""
    nic, njc, nv = q.shape
    B = np.zeros((nic, njc, len(pm.SLOTS), nv, nv))
    I, Jx = np.meshgrid(np.arange(nic), np.arange(njc), indexing="ij")
    for a in range(per):
        for b in range(per):
            on = (I % per == a) & (Jx % per == b)
            for m in range(nv):
                v = np.zeros_like(q)
                v[..., m] = on
                _, jv = of.jv(case, q, v, wd=wd)
                for s, (di, dj) in enumerate(pm.SLOTS):
                    if max(abs(di), abs(dj)) > per // 2:
                        continue
                    ii, jj = I + di, Jx + dj
                    ok = (ii >= 0) & (ii < nic) & (jj >= 0) & (jj < njc) & (ii % per == a) & (jj % per == b)
                    B[:, :, s, :, m][ok] = jv[ok]
    return B


@pytest.mark.parametrize("cols,rows,sa,width", [
    (1024, 5, True, 8),     # 256 groups: still two lanes
    (1025, 9, True, 8),     # one group a chunk, a last chunk of one column
    (1363, 6, True, 16),    # groups of 8; a last chunk of three columns
    (1549, 8, True, 24),    # groups of 12; a last chunk of a group and one column
    (1377, 66, True, 32),   # groups of 11; a last chunk of one column; the ring wraps
    (1388, 3, True, 32),    # a last chunk of a group and one column; three rows
    (2049, 11, False, 8),   # nv = 4: one group a chunk
    (2065, 7, False, 16),   # one group of 16; a last chunk of one column
    (2047, 4, False, 24),   # groups of 12; a last chunk of seven columns
    (2066, 65, False, 32),  # groups of 16; a last chunk of a group and two columns; the ring wraps
])
@pytest.mark.parametrize("precond", [6, 7])
def test_wide_grids_match_model(cols, rows, sa, width, precond):
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
    B = oracle_blocks(cj, q, eq.walldist() if sa else None, 3 if nine else 5)
    nchunk = (cols + width - 1) // width
    spans = [(0, width), (nchunk // 2 * width, nchunk // 2 * width + width), ((nchunk - 2) * width, cols)]
    rng = np.random.default_rng(3)
    for transpose in (False, True):
        v = rng.standard_normal(q.shape)
        eq.ls_precond_apply(rng.standard_normal(q.shape), transpose=transpose)  # leaves nothing for the next apply
        z = eq.ls_precond_apply(v, transpose=transpose)
        for a, b in spans:
            zr = pm.ilu_chunked(B[a:b], 1.0 / dt[a:b, :, 0], v[a:b], width, transpose=transpose, nine_point=nine)
            err = float(np.abs(z[a:b] - zr).max() / np.abs(zr).max())
            print(cols, rows, "sa", sa, "width", width, "precond", precond, "transpose", transpose, "columns", a, b,
                  "err", err, flush=True)
            # the factors are rounded to float32 on both sides from FP64 values
            # that agree to about 1e-12: now and then one lands on the other
            # neighbour, 6e-8 away; a wrong row or column is off by more than 1e-3
            assert err <= 1e-6
    eq.close()
