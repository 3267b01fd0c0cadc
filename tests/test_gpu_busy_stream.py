"""Work queued on the process's default stream does not delay anything that the
library's own streams rely on: buffers are cleared in the order of the kernels that
use them.  Each case runs alone and then behind some 0.1 s of another library's
work on that stream, with the same results."""
import numpy as np
import pytest

import analogsat_amd as A
import oracle as O

pytestmark = pytest.mark.gpu


def steps():
    p = O.fastsat(40000, 170000, 3, 61)
    sat = A.HipSat("f32")
    sat.SetProblem(A.SatProblem(p.literals, p.lengths))
    old, new, d = sat.MakeState(), sat.MakeState(), sat.MakeState()
    old.CopyFrom(np.concatenate([np.random.default_rng(1).uniform(-1, 1, p.n), np.ones(p.m)]).astype(np.float32))

    def go():
        rk = A.HipRungeKutta()
        rk.SetEpsilon(1e-6)
        rk.Configure(sat)
        sat.GetDerivatives(d, old, 0.0)
        assert rk.Step(old, new, 3)
        st = rk.stats()
        assert st.steps == 3
        return old.CopyTo(), d.CopyTo(), st.time, st.hdid, st.attempts
    return go


def few_workgroups():
    p = O.fastsat(2000, 8500, 3, 62)
    sat = A.HipSat("f64")
    sat.SetProblem(A.SatProblem(p.literals, p.lengths))
    old, new = sat.MakeState(), sat.MakeState()
    old.CopyFrom(np.concatenate([np.random.default_rng(2).uniform(-1, 1, p.n), np.ones(p.m)]))

    def go():
        rk = A.HipRungeKutta()
        rk.SetEpsilon(1e-6)
        rk.Configure(sat)
        assert rk.Step(old, new, 5)
        return old.CopyTo(), rk.stats().time, rk.stats().attempts
    return go


def adjoint():
    p = O.fastsat(500, 2100, 3, 63)
    x = np.stack([np.concatenate([np.random.default_rng(i).uniform(-1, 1, p.n), np.ones(p.m)]) for i in range(5)])

    def go():
        a = A.HipAdjoint(A.SatProblem(p.literals, p.lengths), eps=1e-6, steps=12, checkpoint_every=5)
        return a.forward(x.astype(np.float32)), a.backward()
    return go


def batch():
    ps = [O.fastsat(4000, 38000, 4, 64 + i) for i in range(3)]

    def go():
        b = A.HipBatch()
        for i, p in enumerate(ps):
            b.add(A.SatProblem(p.literals, p.lengths),
                  np.concatenate([np.random.default_rng(i).uniform(-1, 1, p.n), np.ones(p.m)]).astype(np.float32))
        b.set_params(eps=1e-6, max_steps=4, chunk_steps=4)
        b.prepare(autotune=False)
        b.run(graph_chunks=1)
        return tuple(b.state(i) for i in range(3)) + tuple(r["attempts"] for r in b.results())
    return go


@pytest.mark.parametrize("case", [steps, few_workgroups, adjoint, batch])
def test_behind_other_work(case):
    A.lib()
    import torch
    x = torch.zeros(1 << 28, device="cuda")
    alone = case()()          # each from its own start
    go = case()
    for _ in range(200):
        x.add_(1.0)
    busy = go()
    assert float(x[0]) == 200.0
    for a, b in zip(alone, busy):
        assert np.array_equal(a, b)
