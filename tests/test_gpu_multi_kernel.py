"""The multi-kernel integrator (tiled clause pass, region var pass, slot spins) on
problems that the persistent kernels would take: 4-literal clauses, rows with padding
slots, and 2048-clause tiles, 30 steps bit for bit against the oracle, also after a
standalone right-hand side (which reuses the contribution array), after the state is
replaced between Steps (the slot spins are made again from it), and when a persistent
kernel has run in between."""
import numpy as np
import pytest

import analogsat_amd as A
import oracle as O

pytestmark = pytest.mark.gpu


def problem(case):
    if case == "k4":
        return O.fastsat(3000, 29700, 4, 5)
    if case == "tiles":
        return O.fastsat(2000, 8500, 3, 33)
    rng = np.random.default_rng(6)
    lens = rng.choice([1, 2, 3], size=9000, p=[0.1, 0.3, 0.6]).astype(np.int32)
    rows = np.argsort(rng.random((9000, 40)), axis=1)[:, :3] + rng.integers(0, 2960, (9000, 1)) + 1
    lits = (rows * rng.choice([-1, 1], (9000, 3))).astype(np.int32)
    return O.Problem(lits[np.arange(3)[None, :] < lens[:, None]], lens)


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("case", ["k4", "mixed", "tiles"])
@pytest.mark.parametrize("between", ["rhs", "replaced", "persistent"])
def test_steps_bitexact(case, precision, between):
    print("[gpu-multi-kernel]", case, precision, between, flush=True)
    p = problem(case)
    mode = "f64" if precision == "f64" else "mix"
    sat = A.HipSat(precision)
    sat.SetProblem(A.SatProblem(p.literals, p.lengths))
    layout = sat.Layout()
    assert layout["clause_pass"] == 0 and layout["var_pass"] == 0 and layout["slot_spins"] == 1
    assert layout["tile_clauses"] == 2048
    rk = A.HipRungeKutta()
    rk.SetEpsilon(1e-6)
    rk.Configure(sat)
    assert rk.Workgroups() >= 8
    rk.SetOneWorkgroup(False)
    old, new = sat.MakeState(), sat.MakeState()
    pub = O.random_state_f64(9, p.n, p.m).astype(sat.dtype)
    old.CopyFrom(pub)
    with O.pow_mode("cr"):
        orc = O.RK(p, eps=1e-6, mode=mode)
        orc.set_state(pub)
        for blk in range(3):
            if blk and between == "rhs":
                d = sat.MakeState()
                sat.GetDerivatives(d, old, 0.0)
            elif blk and between == "replaced":
                moved = old.CopyTo()
                moved[:p.n] = np.clip(moved[:p.n] * sat.dtype(0.5), -1, 1)
                old.CopyFrom(moved)
                orc.set_state(moved)
            elif blk:
                rk.SetOneWorkgroup(True)
                assert rk.Workgroups() >= 8 and rk.Step(old, new, 3)
                orc.step(3)
                rk.SetOneWorkgroup(False)
            assert rk.Step(old, new, 10)
            orc.step(10)
            assert np.array_equal(old.CopyTo(), orc.get_state()), blk
            st = rk.stats()
            assert (st.hdid, st.attempts, st.rhscount) == (orc.hdid, orc.attempts, orc.rhscount), blk
    assert sat.GetClauseViolationCount(old) == orc.violations()
