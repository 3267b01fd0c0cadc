"""Captured attempts between 2^18 literal slots and 4 MiB of contributions, bit for
bit against the oracle: the first Step launches its kernels one by one, the second
one captures them, later ones replay, with a right-hand side, a changed state, other
states and Steps too short for the graph in between; a long first Step captures at
once."""
import numpy as np
import pytest

import analogsat_amd as A
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,n,m,k,counts", [
    ("f64", 30000, 90000, 3, (9, 12, 3, 17, 8, 20)), ("f32", 33000, 90000, 3, (8, 8, 26, 1, 15)),
    ("f32", 5000, 66000, 4, (10, 10, 10)), ("f64", 30000, 90000, 3, (130, 9))])
def test_steps_with_and_without_the_graph(precision, n, m, k, counts):
    p = O.fastsat(n, m, k, 41)
    dt, mode = (np.float64, "f64") if precision == "f64" else (np.float32, "mix")
    sat = A.HipSat(precision)
    sat.SetProblem(A.SatProblem(p.literals, p.lengths))
    rk = A.HipRungeKutta()
    rk.SetEpsilon(1e-6)
    rk.Configure(sat)
    rk.SetOneWorkgroup(False)
    pub = np.concatenate([np.random.default_rng(6).uniform(-1, 1, p.n), np.ones(p.m)]).astype(dt)
    old, new, d = sat.MakeState(), sat.MakeState(), sat.MakeState()
    old.CopyFrom(pub)
    with O.pow_mode("cr"):
        orc = O.RK(p, eps=1e-6, mode=mode)
        orc.set_state(pub)
        for i, count in enumerate(counts):
            print("[gpu-step-graph]", precision, p.n, p.m, k, "Step", i, count, flush=True)
            if i == 2:
                sat.GetDerivatives(d, old, 0.0)
                moved = old.CopyTo()
                moved[:p.n] *= dt(0.5)
                old.CopyFrom(moved)
                orc.set_state(moved)
            if i == 4:
                old2, new = sat.MakeState(), sat.MakeState()
                old2.CopyFrom(old.CopyTo())
                old = old2
            assert rk.Step(old, new, count)
            orc.step(count)
            assert np.array_equal(old.CopyTo(), orc.get_state()), i
            st = rk.stats()
            assert (st.hdid, st.attempts, st.rhscount) == (orc.hdid, orc.attempts, orc.rhscount), i
