"""What follows a wait between work-groups that gave up: with no polls allowed, a
launch's reducing block gives up while the other blocks still run, and their
values stay behind in the slots that it emptied.  Later results may not be made
of them: each is NaN or right, and right again after a call that returned to the
host."""
import ctypes as C

import numpy as np
import pytest

from structured_amd import cases, lib

pytestmark = pytest.mark.gpu


def set_polls(eq, polls):
    assert lib.load().sg_test_wait_polls(eq.h, C.c_int(polls)) == 0


@pytest.fixture
def eq():
    case = cases.laminar_plate(97, 65)
    e = lib.Equation(case)
    yield e
    set_polls(e, -1)
    e.close()


def states(eq):
    return [eq.case.perturbed_state(seed=s, amp=0.01) for s in (1, 2)]


def on_device(eq, q):
    torch = pytest.importorskip("torch")
    aos = torch.from_numpy(np.ascontiguousarray(q).reshape(-1)).to("cuda:0")
    d = torch.zeros(eq.nvar * eq.plane, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    eq.aos_to_soa_dev(aos.data_ptr(), d.data_ptr())
    eq.synchronize()
    return d


def test_norms_after_a_wait_that_gave_up(eq):
    torch = pytest.importorskip("torch")
    qd = [on_device(eq, q) for q in states(eq)]
    rd = torch.zeros_like(qd[0])
    l2 = torch.zeros(eq.nvar, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()

    def norms(k):
        eq.residual_dev_async(qd[k].data_ptr(), rd.data_ptr(), l2.data_ptr())
        eq.synchronize()
        return l2.cpu().numpy()
    ref = norms(1)
    assert np.isfinite(ref).all()
    set_polls(eq, 0)
    assert np.isnan(norms(0)).any()
    set_polls(eq, -1)
    for _ in range(2):
        after = norms(1)
        print("after", after, "right", ref)
        assert np.array_equal(after, ref) or np.isnan(after).all()
    eq.residual_dev(qd[1].data_ptr(), rd.data_ptr())
    assert np.array_equal(norms(1), ref)


def test_explicit_step_after_a_wait_that_gave_up(eq):
    q1, q2 = states(eq)
    d1, d2, d3 = on_device(eq, q1), on_device(eq, q2), on_device(eq, q2)
    ref = eq.step_explicit_dev(d2.data_ptr(), "rk4_jameson", 0.5)
    assert np.isfinite(ref).all()
    set_polls(eq, 0)
    with pytest.raises(lib.SgError):
        eq.step_explicit_dev(d1.data_ptr(), "rk4_jameson", 0.5)
    set_polls(eq, -1)
    assert np.array_equal(eq.step_explicit_dev(d3.data_ptr(), "rk4_jameson", 0.5), ref)


def test_linear_solve_after_a_wait_that_gave_up(eq):
    q1, q2 = states(eq)
    dt = eq.calc_dt(q1, 20.0)
    r1, _ = eq.calc_residual(q1)
    r2, _ = eq.calc_residual(q2)
    eq.ls_preallocate(restart=12, precond=4, maxit=12, rtol=1e-6)
    eq.ls_set_lhs(q1, dt)
    eq.ls_set_rhs(r2)
    ref = eq.ls_solve()
    eq.ls_set_rhs(r1)
    set_polls(eq, 0)
    with pytest.raises(lib.SgError):
        eq.ls_solve()
    set_polls(eq, -1)
    eq.ls_set_rhs(r2)
    got = eq.ls_solve()
    assert got[1:] == ref[1:] and np.array_equal(got[0], ref[0])


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("few", [0, 1])  # a launch for both passes, a launch each
def test_preconditioner_after_a_wait_that_gave_up(eq, transpose, few):
    assert lib.load().sg_test_few_cus(eq.h, C.c_int(few)) == 1 - few
    q, _ = states(eq)
    dt = eq.calc_dt(q, 20.0)
    rng = np.random.default_rng(1)
    v1, v2 = rng.standard_normal(q.shape), rng.standard_normal(q.shape)
    eq.ls_preallocate(restart=4, precond=7, maxit=4, rtol=1e-6)
    eq.ls_set_pc(1, 1.0, 32)
    eq.ls_set_lhs(q, dt)
    eq.ls_set_rhs(v1)
    refs = [eq.ls_precond_apply(v, transpose=transpose) for v in (v1, v2)]

    def apply(n):
        z = eq.ls_precond_apply((v1, v2)[n], transpose=transpose)
        nan, wrong = np.isnan(z), z != refs[n]
        print("NaN", np.count_nonzero(nan), "wrong", np.count_nonzero(wrong & ~nan))
        assert not (wrong & ~nan).any()
        return nan.any()
    set_polls(eq, 0)
    assert apply(0)
    set_polls(eq, -1)
    assert apply(1) and apply(0)
    with pytest.raises(lib.SgError):  # a solve does not take the NaN for the end of its iteration
        eq.ls_solve()
    eq.ls_set_lhs(q, dt)
    assert not apply(0) and not apply(1)
