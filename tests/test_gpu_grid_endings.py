"""The few-workgroup integrator past what one launch takes (4096 attempts), and ending
by step-size underflow: in 8 and more workgroups and in one, bit for bit with the
multi-kernel path."""
import numpy as np
import pytest

import analogsat_amd as A
import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [("f32", 1100, 6000, 8), ("f64", 130, 700, 1)]      # unsatisfiable: no early end


def pair(prec, n, m, workgroups, positive=False):
    p = O.fastsat(n, m, 3, 51)
    if positive:
        p = O.Problem(np.abs(p.literals), p.lengths)     # solved by all true
    assert (p.n, p.m) == (n, m)
    out = []
    for persistent in (True, False):
        sat = A.HipSat(prec)
        sat.SetProblem(A.SatProblem(p.literals, p.lengths))
        rk = A.HipRungeKutta()
        rk.SetEpsilon(1e-6)
        rk.Configure(sat)
        rk.SetOneWorkgroup(persistent)
        assert rk.Workgroups() >= workgroups if persistent else rk.Workgroups() == 0
        old, new = sat.MakeState(), sat.MakeState()
        old.CopyFrom(np.concatenate([np.random.default_rng(5).uniform(-1, 1, p.n), np.ones(p.m)]).astype(sat.dtype))
        out.append((sat, rk, old, new))
    return out


def same(a, b):
    sa, sb = a[1].stats(), b[1].stats()
    for f in ("time", "hdid", "hnext", "errmax", "steps", "attempts", "rhscount"):
        assert getattr(sa, f) == getattr(sb, f), f
    assert np.array_equal(a[2].CopyTo(), b[2].CopyTo())


@pytest.mark.parametrize("prec,n,m,workgroups", SIZES)
def test_long_step(prec, n, m, workgroups):
    a, b = pair(prec, n, m, workgroups)
    for sat, rk, old, new in (a, b):
        assert rk.Step(old, new, 5000)
    assert a[1].stats().attempts > 4096
    same(a, b)


@pytest.mark.parametrize("prec,n,m,workgroups", SIZES)
def test_long_solve(prec, n, m, workgroups):
    """A batch of 3 that the pause between launches cuts, and one it does not."""
    a, b = pair(prec, n, m, workgroups)
    for batch, steps in ((3, 4500), (500, 4500)):
        ends = []
        for sat, rk, old, new in (a, b):
            r = rk.SolveBatches(old, new, batch, steps, 1e300)
            ends.append((r.result, r.steps, r.last_violations))
        assert ends[0] == ends[1]
        assert ends[0][0] == A.SatResult.SAT_MAXITER_REACHED
        same(a, b)


@pytest.mark.parametrize("solve", [False, True])
@pytest.mark.parametrize("n,m,workgroups", [(1100, 6000, 8), (130, 700, 1)])
def test_underflow(n, m, workgroups, solve):
    """At a solution nothing moves and the step grows to 1e15; from states a little
    further off each time it then has to shrink, until it no longer moves the time."""
    a, b = pair("f64", n, m, workgroups, positive=True)
    ends = []
    for sat, rk, old, new in (a, b):
        old.CopyFrom(np.ones(n + m))
        assert rk.Step(old, new, 36)
        assert rk.GetTime() > 1e15
        for i in range(22):
            s = 1 - 1e-4 * 1.5 ** i * np.random.default_rng(3).uniform(0.5, 1, n)
            old.CopyFrom(np.concatenate([s, np.ones(m)]))
            if i < 21:
                assert rk.Step(old, new, 4), i
        if solve:
            r = rk.SolveBatches(old, new, 4, 1000, 1e300)
            ends.append((r.result, r.steps, r.last_violations))
            assert r.result == A.SatResult.SAT_UNDERFLOW
        else:
            assert not rk.Step(old, new, 4)
            ends.append(rk.stats().steps)
        assert not rk.Step(old, new, 1)
    assert ends[0] == ends[1]
    same(a, b)
