"""The few-workgroup integrator where its workgroups are not all resident: a
problem that needs more of them than the device holds takes the multi-kernel path,
and so does one whose workgroups wait in vain, from where its launches stopped.
Results, counters and endings stay those of the multi-kernel path throughout."""
import threading

import numpy as np
import pytest

import analogsat_amd as A
import oracle as O

pytestmark = pytest.mark.gpu


def solver(prec, n, m, seed, **limits):
    p = O.fastsat(n, m, 3, seed)
    sat = A.HipSat(prec)
    sat.SetProblem(A.SatProblem(p.literals, p.lengths))
    rk = A.HipRungeKutta()
    rk.SetEpsilon(1e-6)
    rk.Configure(sat)
    if limits.pop("multi_kernel", False):
        rk.SetOneWorkgroup(False)
    rk.SetGridLimits(**limits)
    old, new = sat.MakeState(), sat.MakeState()
    old.CopyFrom(np.concatenate([np.random.default_rng(seed).uniform(-1, 1, p.n), np.ones(p.m)]).astype(sat.dtype))
    return sat, rk, old, new


def counters(rk):
    st = rk.stats()
    return st.time, st.hdid, st.hnext, st.errmax, st.steps, st.attempts, st.rhscount


# more workgroups than allowed, a wait given up in the first launch, and in one
# after launches that paused
LIMITS = [{"workgroups": 7}, {"launches": 0}, {"attempts": 7, "launches": 2}]


@pytest.mark.parametrize("limits", LIMITS)
@pytest.mark.parametrize("prec,n,m", [("f32", 2000, 8500), ("f64", 5000, 21250)])
def test_steps_go_on_by_the_multi_kernel_path(prec, n, m, limits):
    out = []
    for lim in ({"multi_kernel": True}, dict(limits), {"attempts": 5}):
        sat, rk, old, new = solver(prec, n, m, 31, **lim)
        got = []
        for count in (12, 1, 9):
            assert rk.Step(old, new, count)
            got.append((counters(rk), old.CopyTo()))
        out.append(got)
    for other in out[1:]:
        for (ca, xa), (cb, xb) in zip(out[0], other):
            assert ca == cb
            assert np.array_equal(xa, xb)


@pytest.mark.parametrize("limits", LIMITS)
@pytest.mark.parametrize("m,batch,max_steps,max_time", [
    (4000, 1, 4000, 1e300), (4000, 7, 4000, 1e300), (8500, 5, 33, 1e300), (8500, 4, 4000, 0.3)])
def test_solves_end_the_same(m, batch, max_steps, max_time, limits):
    """SAT, the step limit and the time limit; with limits on the launches, in and between batches."""
    ends = []
    for lim in ({"multi_kernel": True}, dict(limits)):
        sat, rk, old, new = solver("f64", 2000, m, 32, **lim)
        r = rk.SolveBatches(old, new, batch, max_steps, max_time)
        assert r.on_device == 0
        ends.append((r.result, r.steps, r.last_violations, counters(rk), old.CopyTo()))
    assert ends[0][:4] == ends[1][:4]
    assert np.array_equal(ends[0][4], ends[1][4])
    if m == 4000:
        assert ends[0][0] == A.SatResult.SAT_SOLUTION_FOUND


def test_a_small_problem_goes_on_in_one_workgroup():
    """More than 1024 variables, but small enough for the one-workgroup kernel: its
    launches take over, also in the middle of a solve."""
    ends = []
    for lim in ({"multi_kernel": True}, {"attempts": 6, "launches": 3}, {}):
        sat, rk, old, new = solver("f32", 1100, 1500, 33, **lim)
        r = rk.SolveBatches(old, new, 3, 60, 1e300)
        assert r.on_device == (0 if "multi_kernel" in lim else 1)
        ends.append((r.result, r.steps, r.last_violations, counters(rk), old.CopyTo()))
    for other in ends[1:]:
        assert ends[0][:4] == other[:4]
        assert np.array_equal(ends[0][4], other[4])


def test_another_problem_is_tried_again():
    sat, rk, old, new = solver("f64", 2000, 8500, 34, launches=0)
    assert rk.SolveBatches(old, new, 5, 20, 1e300).on_device == 0
    rk.SetGridLimits()
    assert rk.SolveBatches(old, new, 5, 20, 1e300).on_device == 0
    p = O.fastsat(2000, 8500, 3, 35)
    sat.SetProblem(A.SatProblem(p.literals, p.lengths))
    rk.Configure(sat)
    old, new = sat.MakeState(), sat.MakeState()
    old.CopyFrom(np.concatenate([np.zeros(p.n) + 0.1, np.ones(p.m)]))
    assert rk.SolveBatches(old, new, 5, 20, 1e300).on_device == 1


@pytest.mark.parametrize("prec,n,m", [("f32", 2000, 8500), ("f64", 12000, 51120)])
def test_two_integrators_from_two_threads(prec, n, m):
    def go(seed, out):
        sat, rk, old, new = solver(prec, n, m, seed)
        for _ in range(6):
            assert rk.Step(old, new, 10)
        out[seed] = (counters(rk), old.CopyTo())

    alone, both = {}, {}
    for seed in (36, 37):
        go(seed, alone)
    threads = [threading.Thread(target=go, args=(seed, both)) for seed in (36, 37)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for seed in (36, 37):
        assert alone[seed][0] == both[seed][0]
        assert np.array_equal(alone[seed][1], both[seed][1])
