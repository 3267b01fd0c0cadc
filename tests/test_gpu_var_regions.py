"""LDS var pass on groups with more 16-byte units than a workgroup reads in one
round (FP32: 16 384 contributions, FP64: 12 288), bit for bit against the oracle:
with slot spins and direct primary terms (3 and 4 literals) and without (5), a
group of one unit more and one near the largest."""
import numpy as np
import pytest

import analogsat_amd as A
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,k,m", [
    ("f32", 3, 5462), ("f32", 3, 8100), ("f32", 4, 6001), ("f32", 5, 4801),
    ("f64", 3, 4097), ("f64", 3, 4801), ("f64", 4, 3601), ("f64", 5, 2881)])
def test_regions_of_several_rounds(precision, k, m):
    print("[gpu-var-regions]", precision, k, m, flush=True)
    n = 101
    rng = np.random.default_rng(m)
    rows = np.argsort(rng.random((m, n)), axis=1)[:, :k] + 1
    rows[0] = np.arange(n - k + 1, n + 1)
    lits = (rows * rng.choice([-1, 1], (m, k))).astype(np.int32)
    p = O.Problem(lits.reshape(-1), np.full(m, k, np.int32))
    dt, mode = (np.float64, "f64") if precision == "f64" else (np.float32, "mix")
    sat = A.HipSat(precision)
    sat.SetProblem(A.SatProblem(p.literals, p.lengths))
    layout = sat.Layout()
    assert layout["var_pass"] == 0 and layout["groups"] == 1
    pub = np.concatenate([rng.uniform(-1, 1, p.n), np.ones(p.m)]).astype(dt)
    x, d = sat.MakeState(), sat.MakeState()
    x.CopyFrom(pub)
    sat.GetDerivatives(d, x, 0.0)
    assert np.array_equal(d.CopyTo(), O.rhs(p, np.concatenate([[-1.0], pub]).astype(dt), mode=mode)[1:])
    rk = A.HipRungeKutta()
    rk.SetEpsilon(1e-6)
    rk.Configure(sat)
    rk.SetOneWorkgroup(False)
    old, new = sat.MakeState(), sat.MakeState()
    old.CopyFrom(pub)
    with O.pow_mode("cr"):
        orc = O.RK(p, eps=1e-6, mode=mode)
        orc.set_state(pub)
        for count in (2, 10):
            rk.Step(old, new, count)
            orc.step(count)
            assert np.array_equal(old.CopyTo(), orc.get_state())
        st = rk.stats()
        assert (st.hdid, st.attempts, st.rhscount) == (orc.hdid, orc.attempts, orc.rhscount)
