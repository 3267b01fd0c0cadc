"""States read from another thread while a batch runs: each one is whole (the state
of the latest finished launch), and none of them is served again after the run."""
import threading

import numpy as np
import pytest

import analogsat_amd as A
import oracle as O

pytestmark = pytest.mark.gpu

STEPS = 3000


def batch():
    b = A.HipBatch()
    for i in range(40):
        p = O.fastsat(60 + i, 6 * (60 + i), 3, 300 + i)      # far above the threshold: no early end
        b.add(A.SatProblem(p.literals, p.lengths),
              np.concatenate([np.random.default_rng(i).uniform(-1, 1, p.n), np.ones(p.m)]).astype(np.float32))
    b.set_params(eps=1e-6, max_steps=STEPS, chunk_steps=1, check_every=1)
    b.set_tiling(block=256, lds_mode=2, nbuckets=2)
    b.prepare(autotune=False)
    return b


def test_states_read_beside_a_run():
    alone = batch()
    alone.run(graph_chunks=1)
    want = [alone.state(i) for i in range(len(alone))]
    b = batch()
    worker = threading.Thread(target=b.run, kwargs={"graph_chunks": 1})
    worker.start()
    while b.result(0)["steps"] == 0 and worker.is_alive():
        pass
    early = [b.state(i) for i in range(len(b))]
    steps = b.result(0)["steps"]
    worker.join()
    print("[gpu-batch-threads] states read at step", steps, flush=True)
    assert 0 < steps < STEPS
    assert all(np.isfinite(x).all() for x in early)
    for i in range(1, len(b)):
        assert np.array_equal(b.state(i), want[i]), i
    assert any(not np.array_equal(early[i], want[i]) for i in range(1, len(b)))
