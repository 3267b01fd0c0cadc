"""The few-workgroup persistent integrator (problems between one workgroup's LDS
and the multi-kernel path): states, step sizes and counters equal the
multi-kernel path's (forced with SetOneWorkgroup(False)) and the oracle's, at
the edges of its layout: whole groups of 64 variables and one more, clause
lists just filling and overflowing a thread's registers, short clauses, the
largest problems it takes and the first ones past it, and every way a solve
can end.
"""
import numpy as np
import pytest

import analogsat_amd as A
import oracle as O

pytestmark = pytest.mark.gpu


def make(n, m, k, seed, short=0.0):
    p = O.fastsat(n, m, k, seed)
    if short:
        rng = np.random.default_rng(seed)
        keep = np.ones((m, k), bool)
        keep[1:, k - 1] = rng.random(m - 1) >= short
        keep[2::7, 1:] = False                       # one-literal clauses too
        p = O.Problem(p.literals.reshape(m, k)[keep].astype(np.int32), keep.sum(1).astype(np.int32))
    return p


def start(p, prec, seed=8):
    s = np.random.default_rng(seed).uniform(-1, 1, p.n)
    s[::17] = 0.0
    return np.concatenate([s, np.ones(p.m)]).astype(np.float64 if prec == "f64" else np.float32)


def solver(p, prec, persistent, eps=1e-6):
    sat = A.HipSat(prec)
    sat.SetProblem(A.SatProblem(p.literals, p.lengths))
    rk = A.HipRungeKutta()
    rk.SetEpsilon(eps)
    rk.Configure(sat)
    rk.SetOneWorkgroup(persistent)
    assert not (persistent and rk.UsesOneWorkgroup())
    return sat, rk


def run(p, prec, persistent, pub, blocks):
    sat, rk = solver(p, prec, persistent)
    old, new = sat.MakeState(), sat.MakeState()
    old.CopyFrom(pub)
    out = []
    for count in blocks:
        assert rk.Step(old, new, count)
        st = rk.stats()
        out.append((old.CopyTo(), st.time, st.hdid, st.hnext, st.errmax, st.steps, st.attempts, st.rhscount))
    out.append(sat.GetClauseViolationCount(old))
    return out


def same(a, b):
    for i, (x, y) in enumerate(zip(a[:-1], b[:-1])):
        assert x[1:] == y[1:], i
        assert np.array_equal(x[0], y[0]), i
    assert a[-1] == b[-1]


@pytest.mark.parametrize("prec,n,m,k,short", [
    ("f64", 640, 2700, 3, 0.0), ("f64", 641, 2700, 3, 0.3), ("f32", 1023, 4300, 3, 0.2), ("f32", 1025, 9000, 4, 0.3),
    ("f64", 200, 1990, 4, 0.0), ("f32", 5000, 21250, 3, 0.0), ("f64", 6000, 59000, 4, 0.0),
    ("f64", 12000, 51120, 3, 0.1), ("f64", 19900, 60000, 3, 0.0), ("f64", 19968, 60000, 3, 0.0),
    ("f32", 24000, 102000, 3, 0.0), ("f32", 32700, 120000, 3, 0.0), ("f32", 900, 70000, 3, 0.0)])
def test_steps_equal_the_multi_kernel_path(prec, n, m, k, short):
    p = make(n, m, k, 5, short)
    pub = start(p, prec)
    same(run(p, prec, True, pub, (1, 9, 8)), run(p, prec, False, pub, (1, 9, 8)))


@pytest.mark.parametrize("prec,mode", [("f64", "f64"), ("f32", "mix")])
def test_steps_equal_the_oracle(prec, mode):
    p = make(700, 2900, 3, 6, short=0.2)
    pub = start(p, prec)
    got = run(p, prec, True, pub, (7, 20))
    with O.pow_mode("cr"):
        orc = O.RK(p, eps=1e-6, mode=mode)
        orc.set_state(pub)
        for i, count in enumerate((7, 20)):
            orc.step(count)
            assert np.array_equal(got[i][0], orc.get_state()), i
            assert got[i][2] == orc.hdid and got[i][6] == orc.attempts and got[i][7] == orc.rhscount
    assert got[-1] == orc.violations()


@pytest.mark.parametrize("m,batch,max_steps,max_time", [
    (2000, 1, 4000, 1e300), (2000, 7, 4000, 1e300), (2800, 5, 23, 1e300), (2800, 4, 4000, 0.5)])
def test_solve_ends_like_the_host_loop(m, batch, max_steps, max_time):
    """SAT, the step limit and the time limit, with the counts of every ending."""
    p = make(650, m, 3, 11)
    pub = start(p, "f64")
    ends = []
    for persistent in (True, False):
        sat, rk = solver(p, "f64", persistent)
        old, new = sat.MakeState(), sat.MakeState()
        old.CopyFrom(pub)
        r = rk.SolveBatches(old, new, batch, max_steps, max_time)
        st = rk.stats()
        assert r.on_device == int(persistent)
        ends.append((r.result, r.steps, r.last_violations, st.time, st.attempts, old.CopyTo()))
    assert ends[0][:5] == ends[1][:5]
    assert np.array_equal(ends[0][5], ends[1][5])
    if m == 2000:
        assert ends[0][0] == A.SatResult.SAT_SOLUTION_FOUND


@pytest.mark.parametrize("prec,n,m,k,short", [
    ("f64", 120, 513, 3, 0.0), ("f64", 64, 600, 4, 0.3), ("f64", 65, 1024, 3, 0.2), ("f64", 500, 2048, 3, 0.0),
    ("f32", 1024, 4096, 3, 0.1), ("f32", 513, 300, 3, 0.0), ("f32", 400, 3972, 4, 0.2)])
def test_one_workgroup_with_state_in_registers(prec, n, m, k, short):
    """One workgroup of 1024 threads: from 513 clauses or variables on, up to what
    its threads hold."""
    p = make(n, m, k, 12, short)
    pub = start(p, prec)
    out = []
    for persistent in (True, False):
        sat = A.HipSat(prec)
        sat.SetProblem(A.SatProblem(p.literals, p.lengths))
        rk = A.HipRungeKutta()
        rk.SetEpsilon(1e-6)
        rk.Configure(sat)
        rk.SetOneWorkgroup(persistent)
        old, new = sat.MakeState(), sat.MakeState()
        old.CopyFrom(pub)
        assert rk.Step(old, new, 23)
        r = rk.SolveBatches(old, new, 3, 31, 1e300)
        st = rk.stats()
        out.append((r.result, r.steps, r.last_violations, st.time, st.hdid, st.hnext, st.attempts, st.rhscount,
                    old.CopyTo()))
    assert out[0][:-1] == out[1][:-1]
    assert np.array_equal(out[0][-1], out[1][-1])
