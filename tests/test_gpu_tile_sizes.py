"""Clause tiles of fewer than 2048 clauses, bit for bit against the oracle: below
and at the smallest number of clauses that gets them, the smallest tiles, tiles of
one clause more than a workgroup has threads for at a time, two rounds of tiles, a
last tile that is partly empty, and clauses shorter than the longest one."""
import numpy as np
import pytest

import analogsat_amd as A
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,k,m,tile", [
    ("f64", 3, 32767, 2048), ("f64", 3, 32768, 512), ("f64", 3, 131073, 576), ("f64", 3, 262145, 1088),
    ("f64", 3, 530001, 1088), ("f64", 4, 33001, 512), ("f32", 4, 32768, 512), ("f32", 4, 200003, 832)])
def test_tile_sizes(precision, k, m, tile):
    print("[gpu-tile-sizes]", precision, k, m, flush=True)
    n = max(12001, m // 5)
    rng = np.random.default_rng(m)
    first = rng.integers(1, n + 1, m)
    rows = (first[:, None] - 1 + np.cumsum(rng.integers(0, n // (k + 1), (m, k)) + 1, axis=1)) % n + 1
    lits = (rows * rng.choice([-1, 1], (m, k))).astype(np.int32)
    lens = np.where(rng.random(m) < 0.1, k - 1, k).astype(np.int32)
    lens[0] = k
    p = O.Problem(lits[np.arange(k)[None, :] < lens[:, None]], lens)
    dt, mode = (np.float64, "f64") if precision == "f64" else (np.float32, "mix")
    sat = A.HipSat(precision)
    sat.SetProblem(A.SatProblem(p.literals, p.lengths))
    assert sat.Layout()["tile_clauses"] == tile
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
        rk.Step(old, new, 4)
        orc.step(4)
        assert np.array_equal(old.CopyTo(), orc.get_state())
