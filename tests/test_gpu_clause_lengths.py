"""Clause lengths outside the tiled pass (other than 3 and 4), bit for bit against
the oracle: each compile-time bound of the generic clause pass at and below its
length, clauses shorter than the longest one, a last workgroup that is partly
empty, sparse problems (LDS var pass) and dense ones (a variable's contributions
side by side, rows that end inside a batch and just past a chunk)."""
import numpy as np
import pytest

import analogsat_amd as A
import oracle as O

pytestmark = pytest.mark.gpu


def problem(n, m, k, seed):
    rng = np.random.default_rng(seed)
    lens = rng.integers(max(1, k - 2), k + 1, m).astype(np.int32)
    lens[0] = k
    rows = np.argsort(rng.random((m, n)), axis=1)[:, :k] + 1 if n <= 64 else rng.integers(1, n + 1, (m, k))
    if n > 64:
        for j in range(m):
            rows[j] = rng.choice(n, k, replace=False) + 1
    lits = (rows * rng.choice([-1, 1], (m, k))).astype(np.int32)
    return O.Problem(lits[np.arange(k)[None, :] < lens[:, None]], lens)


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("n,m,k", [
    (700, 1500, 1), (700, 1500, 2), (700, 2049, 5), (700, 2048, 6), (500, 1000, 7), (500, 1001, 8), (400, 900, 9),
    (400, 900, 10), (300, 700, 11), (40, 6144, 5), (40, 30000, 6), (30, 12289, 10)])
def test_clause_lengths(n, m, k, precision):
    p = problem(n, m, k, 100 * k + n)
    dt, mode = (np.float64, "f64") if precision == "f64" else (np.float32, "mix")
    sat = A.HipSat(precision)
    sat.SetProblem(A.SatProblem(p.literals, p.lengths))
    pub = np.concatenate([np.random.default_rng(k).uniform(-1, 1, p.n), np.ones(p.m)]).astype(dt)
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
        for count in (3, 12):
            rk.Step(old, new, count)
            orc.step(count)
            assert np.array_equal(old.CopyTo(), orc.get_state())
        st = rk.stats()
        assert (st.hdid, st.attempts, st.rhscount) == (orc.hdid, orc.attempts, orc.rhscount)
    assert sat.GetClauseViolationCount(old) == orc.violations()
