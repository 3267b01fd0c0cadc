"""Adjoint runs whose trajectories share tiles: every trajectory's steps, V, end
state and gradient are those of a run of its own, bit for bit (the sums of a
trajectory run in the same order for every number of trajectories), at numbers
of trajectories that leave tiles and XCDs part empty, and with clauses of
several lengths; and a second run in the same object, whose buffers are kept,
and one after a change of sizes, whose buffers are not."""
import sys

import numpy as np
import pytest

import analogsat_amd as A
import oracle as O

pytestmark = pytest.mark.gpu


def problem(k, n, m, seed):
    p = O.fastsat(n, m, k, seed)
    if k == 3:
        return A.SatProblem(p.literals, p.lengths)
    rng = np.random.default_rng(seed)
    lits, lens, at = [], [], 0
    for j, ln in enumerate(p.lengths):
        keep = int(ln) if j == 0 else int(rng.integers(2, ln + 1))
        lits.extend(p.literals[at:at + keep])
        lens.append(keep)
        at += int(ln)
    return A.SatProblem(np.asarray(lits, np.int32), np.asarray(lens, np.int32))


def starts(sp, ntraj, seed):
    rng = np.random.default_rng(seed)
    n, m = int(np.abs(sp.literals).max()), len(sp.lengths)
    return np.concatenate([rng.uniform(-1, 1, (ntraj, n)), rng.uniform(1, 2, (ntraj, m))], axis=1).astype(np.float32)


@pytest.mark.parametrize("ntraj", [9, 20, 67])
@pytest.mark.parametrize("k,n,m", [(3, 61, 257), (4, 33, 300)])
def test_tiles_do_not_change_a_trajectory(k, n, m, ntraj):
    check(k, n, m, ntraj)


# more slots than the 2^16 up to which a tile has 8 trajectories at most: five
# tiles of one, two of 16 (four XCDs each), one of four (all XCDs)
@pytest.mark.parametrize("ntraj", [5, 31, 4])
def test_large_problem_tiles(ntraj):
    check(3, 5001, 22001, ntraj, T=3)


def check(k, n, m, ntraj, T=12):
    print("[gpu-adjoint-tiles]", k, n, m, ntraj, flush=True)
    sys.stdout.flush()
    sp = problem(k, n, m, 11 * k + n)
    pubs = starts(sp, ntraj, ntraj)
    adj = A.HipAdjoint(sp, eps=1e-6, steps=T, checkpoint_every=5)
    V, h = adj.forward(pubs), adj.steps()
    g = adj.backward()
    Vr, xT = adj.replay(pubs, h)
    assert np.array_equal(Vr, V)
    Vd = adj.replay_f64(pubs.astype(np.float64), h)
    one = A.HipAdjoint(sp, eps=1e-6, steps=T, checkpoint_every=5)
    for t in sorted({0, 1, min(7, ntraj - 1), ntraj // 2, ntraj - 1}):
        row = pubs[t:t + 1]
        assert one.forward(row)[0] == V[t]
        assert np.array_equal(one.steps()[0], h[t])
        assert np.array_equal(one.backward()[0], g[t])
        _, x1 = one.replay(row, h[t:t + 1])
        assert np.array_equal(x1[0], xT[t])
        assert one.replay_f64(row.astype(np.float64), h[t:t + 1])[0] == Vd[t]


def test_buffers_kept_and_changed():
    print("[gpu-adjoint-tiles] kept buffers", flush=True)
    sp = problem(3, 61, 257, 5)
    a, b = starts(sp, 17, 1), starts(sp, 17, 2)
    adj = A.HipAdjoint(sp, eps=1e-6, steps=10, checkpoint_every=4)
    Va, ga = adj.forward(a), adj.backward()
    adj.forward(b)
    adj.backward()
    V5 = adj.forward(b[:5])
    g5 = adj.backward()
    assert np.array_equal(adj.forward(a), Va)
    assert np.array_equal(adj.backward(), ga)
    new = A.HipAdjoint(sp, eps=1e-6, steps=10, checkpoint_every=4)
    assert np.array_equal(new.forward(b[:5]), V5)
    assert np.array_equal(new.backward(), g5)
