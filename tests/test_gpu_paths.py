"""Which integrator runs: the number of workgroups that the query reports, for sizes
on both sides of each rule and for the settings that rule a path out."""
import os
import subprocess
import sys
import threading

import numpy as np
import pytest

import analogsat_amd as A

pytestmark = pytest.mark.gpu


def configured(prec, n, m, k=3, family="ctds"):
    sat = A.HipSatTanh(prec) if family == "tanh" else A.HipSat(prec)
    sat.SetProblem(A.fastsat(n, m, k, 2))
    rk = A.HipRungeKutta()
    rk.Configure(sat)
    return sat, rk


@pytest.mark.parametrize("prec,n,m,k,fewest,most,one", [
    ("f64", 50, 213, 3, 1, 1, True), ("f64", 200, 852, 3, 1, 1, True),      # fits one workgroup's LDS
    ("f64", 450, 1900, 3, 1, 1, False), ("f64", 200, 1990, 4, 1, 1, False),  # one workgroup, state in registers
    ("f32", 1100, 1500, 3, 8, 128, False),                                  # fits that LDS, but runs in eight
    ("f64", 650, 2800, 3, 8, 128, False), ("f32", 24000, 102000, 3, 8, 128, False),
    ("f64", 30000, 127500, 3, 0, 0, False), ("f64", 20, 600, 5, 1, 1, True)])
def test_workgroups(prec, n, m, k, fewest, most, one):
    sat, rk = configured(prec, n, m, k)
    print("[gpu-paths]", prec, n, m, k, rk.Workgroups(), flush=True)
    assert fewest <= rk.Workgroups() <= most
    assert rk.UsesOneWorkgroup() == one
    rk.SetOneWorkgroup(False)
    assert rk.Workgroups() == 0 and not rk.UsesOneWorkgroup()


def test_settings_that_rule_a_path_out():
    sat, rk = configured("f64", 2000, 8500)
    assert rk.Workgroups() >= 8
    rk.SetGridLimits(workgroups=7)
    assert rk.Workgroups() == 0
    rk.SetGridLimits()
    assert rk.Workgroups() >= 8
    sat.Set_B(2.0)
    assert rk.Workgroups() == 0
    sat.Set_B(0.0)
    assert rk.Workgroups() >= 8
    assert configured("f64", 2000, 8500, family="tanh")[1].Workgroups() == 0
    assert configured("f64", 50, 213, family="tanh")[1].Workgroups() == 1


def stepped(sat, rk):
    old, new = sat.MakeState(), sat.MakeState()
    old.CopyFrom(np.concatenate([np.random.default_rng(3).uniform(-1, 1, sat.Get_N()),
                                 np.ones(sat.Get_M())]).astype(sat.dtype))
    assert rk.Step(old, new, 12)
    return old.CopyTo(), rk.stats().attempts


def test_a_path_chosen_after_configure():
    """The few-workgroup layout is made when an integrator can first use it: here
    by the setting after Configure, by the family, and by two integrators of one
    system from two threads."""
    sat = A.HipSat("f32")
    sat.SetProblem(A.fastsat(2000, 8500, 3, 2))
    rk = A.HipRungeKutta()
    rk.SetEpsilon(1e-6)
    rk.SetOneWorkgroup(False)
    rk.Configure(sat)
    assert rk.Workgroups() == 0
    want = stepped(sat, rk)
    rk.Reset()
    rk.SetOneWorkgroup(True)
    got = stepped(sat, rk)
    assert rk.Workgroups() >= 8
    assert np.array_equal(got[0], want[0]) and got[1] == want[1]

    sat = A.HipSat("f32")
    sat.SetProblem(A.fastsat(2000, 8500, 3, 2))
    seen = {}

    def configure(i):
        rk = A.HipRungeKutta()
        rk.SetEpsilon(1e-6)
        rk.Configure(sat)
        seen[i] = rk

    threads = [threading.Thread(target=configure, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for rk in seen.values():
        got = stepped(sat, rk)
        assert rk.Workgroups() >= 8
        assert np.array_equal(got[0], want[0]) and got[1] == want[1]


@pytest.mark.parametrize("prec,n,m,k", [
    ("f32", 32700, 120000, 3), ("f64", 17000, 40000, 3), ("f32", 20000, 60000, 3), ("f64", 8000, 79000, 4)])
def test_short_steps_long_steps_and_solves(prec, n, m, k):
    """Near the end of the few-workgroup path's sizes its calls go by their length:
    short Steps by the multi-kernel path, long ones by either, solves of short
    batches on the device.  A mixture of them equals the multi-kernel path alone."""
    p = A.fastsat(n, m, k, 4)
    out = []
    for persistent in (True, False):
        sat = A.HipSat(prec)
        sat.SetProblem(p)
        rk = A.HipRungeKutta()
        rk.SetEpsilon(1e-6)
        rk.Configure(sat)
        rk.SetOneWorkgroup(persistent)
        assert rk.Workgroups() >= 8 if persistent else rk.Workgroups() == 0
        old, new = sat.MakeState(), sat.MakeState()
        old.CopyFrom(np.concatenate([np.random.default_rng(3).uniform(-1, 1, sat.Get_N()),
                                     np.ones(sat.Get_M())]).astype(sat.dtype))
        got = []
        for count in (1, 30, 2):
            assert rk.Step(old, new, count)
            r = rk.SolveBatches(old, new, 2, 5, 1e300)
            assert r.on_device == int(persistent)
            st = rk.stats()
            got.append((r.result, r.steps, r.last_violations, st.time, st.hdid, st.hnext, st.attempts, st.rhscount,
                        old.CopyTo()))
        out.append(got)
    for a, b in zip(*out):
        assert a[:-1] == b[:-1]
        assert np.array_equal(a[-1], b[-1])


@pytest.mark.parametrize("first", ["import torch", "pass"])
def test_second_process(first):
    """A process beside this one, which holds the runtime's one cooperative queue
    of the GPU; also with torch imported between loading the library and its first
    GPU call, where the runtime's occupancy query finds no room for 1024 threads."""
    sat, rk = configured("f32", 2000, 8500)
    want = stepped(sat, rk)
    code = '''
import sys, threading
sys.path.insert(0, %r)
import numpy as np
import analogsat_amd as A
A.lib()
%s
out = {}
def go(i, persistent):
    sat = A.HipSat("f32")
    sat.SetProblem(A.fastsat(2000, 8500, 3, 2))
    rk = A.HipRungeKutta()
    rk.Configure(sat)
    rk.SetOneWorkgroup(persistent)
    assert (rk.Workgroups() >= 8) == persistent, rk.Workgroups()
    old, new = sat.MakeState(), sat.MakeState()
    old.CopyFrom(np.concatenate([np.random.default_rng(3).uniform(-1, 1, sat.Get_N()), np.ones(sat.Get_M())]).astype("f4"))
    assert rk.Step(old, new, 20)
    r = rk.SolveBatches(old, new, 5, 20, 1e300)
    assert r.on_device == int(persistent), r.on_device
    out[i] = old.CopyTo()
go(0, False)
go(1, True)
threads = [threading.Thread(target=go, args=(i, True)) for i in (2, 3)]
for t in threads: t.start()
for t in threads: t.join()
assert all(np.array_equal(out[0], out[i]) for i in (1, 2, 3))
print("same")
''' % (os.path.dirname(os.path.dirname(os.path.abspath(A.__file__))), first)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=180)
    assert r.returncode == 0 and "same" in r.stdout, r.stdout + r.stderr
    rk.Reset()
    again = stepped(sat, rk)
    assert np.array_equal(want[0], again[0]) and want[1] == again[1]
