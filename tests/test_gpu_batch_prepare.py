"""What prepare() builds for each kernel, from several host threads, bit for bit
against the oracle: batches whose buckets take different kernels, a workgroup size
that rules the register kernel out, enough instances for every thread, and prepare()
again after the tiling changed."""
import pytest

import analogsat_amd as A

from test_gpu_batch import check_against_oracle
from test_gpu_batch_layouts import instance

pytestmark = pytest.mark.gpu


def batch(insts, steps):
    b = A.HipBatch()
    for p, pub in insts:
        b.add(A.SatProblem(p.literals, p.lengths), pub)
    b.set_params(eps=1e-6, max_steps=steps, chunk_steps=4, check_every=1)
    return b


@pytest.mark.parametrize("autotune", [False, True])
@pytest.mark.parametrize("sizes,block,nbuckets,modes", [
    ([(700, 3000, 3)] * 2 + [(690, 2900, 3)], 256, 1, {1}),                  # no 256-thread variant: terms in LDS
    ([(5000, 40000, 4)] * 2 + [(60, 250, 3)] * 3, 0, 2, {2, 3}),             # chunked and in registers
    ([(40 + i, 150 + 3 * i, 3) for i in range(300)], 0, 3, {2})])
def test_prepare(sizes, block, nbuckets, modes, autotune):
    insts = [instance(n, m, k, 200 + i, short=0.2 if i % 5 == 1 else 0.0) for i, (n, m, k) in enumerate(sizes)]
    b = batch(insts, 6)
    b.set_tiling(block=block, lds_mode=-1, nbuckets=nbuckets)
    b.prepare(autotune=autotune)
    assert {x["lds"] for x in b.buckets()} == modes, b.buckets()
    b.run(graph_chunks=2)
    check_against_oracle(b, insts, 6)


def test_prepare_again_for_other_kernels():
    insts = [instance(300 + 10 * i, 1200 + 40 * i, 3, 500 + i) for i in range(6)]
    b = batch(insts, 8)
    for mode in (2, 1, 3, 0, -1):
        b.set_tiling(block=0, lds_mode=mode, nbuckets=2)
        b.prepare(autotune=mode == -1)
        assert all(x["lds"] == (2 if mode == -1 else mode) for x in b.buckets()), b.buckets()
        b.run(graph_chunks=2)
        check_against_oracle(b, insts, 8)
