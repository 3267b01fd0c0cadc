"""Batched kernels at the edges of their layouts, bit for bit against the oracle.

Register-resident variants: instances at both ends of what a variant holds
(clauses and variables per thread, whole groups of 64 and one past them, the
two constant ranks at a group's end), clauses shorter than the longest one,
k = 1, 2 and 4, spins of exactly 0 and of a size that leaves 1 - s at 1 (the
violation count then looks at the spin itself).  Clause-chunked kernel: one
clause per chunk more and less than the LDS takes, k = 2, one chunk, many.
"""
import numpy as np
import pytest

import analogsat_amd as A
import oracle as O

from test_gpu_batch import check_against_oracle

pytestmark = pytest.mark.gpu


def instance(n, m, k, seed, short=0.0, tiny=False):
    rng = np.random.default_rng(seed)
    p = O.fastsat(n, m, k, seed)
    lits, lens = p.literals.copy(), p.lengths.copy()
    if short:
        cut = (rng.random(m) < short) & (np.arange(m) > 0) if k > 1 else np.zeros(m, bool)
        rows = lits.reshape(m, k)
        lens = np.where(cut, k - 1, k).astype(np.int32)
        lits = rows[np.arange(k)[None, :] < lens[:, None]].astype(np.int32)
        p = O.Problem(lits, lens)
    pub = np.concatenate([rng.uniform(-1, 1, p.n), np.ones(p.m)]).astype(np.float32)
    if tiny:
        pub[0:p.n:3] = 0.0
        pub[1:p.n:3] = 1e-9
        pub[2:p.n:6] = -1e-9
    return p, pub


def run(insts, steps, block, mode, chunk=0, nbuckets=1):
    b = A.HipBatch()
    for p, pub in insts:
        b.add(A.SatProblem(p.literals, p.lengths), pub)
    b.set_params(eps=1e-6, max_steps=steps, chunk_steps=5, check_every=1)
    b.set_tiling(block=block, lds_mode=mode, nbuckets=nbuckets)
    b.set_chunk(chunk)
    b.prepare(autotune=False)
    assert all(x["lds"] == mode for x in b.buckets()), b.buckets()
    b.run(graph_chunks=2)
    check_against_oracle(b, insts, steps)


# sizes that select each variant in turn: (threads, clauses, variables) per trajectory
@pytest.mark.parametrize("n,m,k,block", [
    (62, 256, 3, 256), (63, 257, 3, 256), (126, 512, 4, 256), (127, 200, 3, 256), (254, 256, 3, 256),
    (255, 1000, 4, 256), (510, 1024, 3, 256), (2046, 4096, 3, 512), (2046, 8704, 3, 512), (2046, 9216, 3, 1024),
    (2047, 8300, 3, 1024), (2048, 8300, 3, 512), (2302, 9000, 3, 0), (2560, 9900, 3, 1024), (2500, 9900, 3, 512),
    (5, 8, 1, 256), (40, 60, 2, 256), (700, 6700, 4, 0), (1, 1, 1, 256)])
def test_register_variants(n, m, k, block):
    insts = [instance(n, m, k, 50 + i, short=0.3 if i == 1 else 0.0, tiny=i == 2) for i in range(3)]
    run(insts, 14, block, 2)


def test_register_variant_mixed_lengths_one_bucket():
    """3-literal, 2-literal and 4-literal instances of one bucket share a kernel for four."""
    run([instance(90, 300, 3, 1), instance(80, 120, 2, 2, short=0.5), instance(70, 500, 4, 3, short=0.5, tiny=True),
         instance(20, 30, 1, 4)], 20, 256, 2)


@pytest.mark.parametrize("n,m,k,block,chunk", [
    (300, 1279, 3, 256, 0), (300, 640, 4, 1024, 320), (300, 641, 4, 512, 320), (65, 130, 2, 256, 64),
    (64, 100, 1, 256, 1), (3000, 12000, 3, 1024, 0), (8100, 30000, 3, 1024, 0), (4100, 40000, 4, 512, 0)])
def test_chunked_layouts(n, m, k, block, chunk):
    insts = [instance(n, m, k, 70 + i, short=0.3 if i == 1 else 0.0, tiny=i == 1) for i in range(2)]
    run(insts, 6, block, 3, chunk=chunk)


def test_states_in_any_order_and_after_every_change():
    """state(i) in order (packed windows) and out of order (single copies) agree
    with each other and follow every run and reset; states of different parity
    and sizes, a window that ends inside the batch."""
    sizes = [(20 + 7 * (i % 5), 60 + 11 * (i % 7)) for i in range(30)] + [(8000, 34000)] * 30   # 1.3e6 floats
    insts = [instance(n, m, 3, 90 + i) for i, (n, m) in enumerate(sizes)]
    b = A.HipBatch()
    for p, pub in insts:
        b.add(A.SatProblem(p.literals, p.lengths), pub)
    b.set_params(eps=1e-6, max_steps=30, chunk_steps=1)
    b.set_tiling(block=256, lds_mode=-1, nbuckets=3)
    b.prepare(autotune=False)
    count = len(insts)
    seen = []
    for limit in (0, 1, 2):
        if limit:
            b.run(max_chunks=1, graph_chunks=1)
        inorder = [b.state(i) for i in range(count)]
        backward = [b.state(i) for i in reversed(range(count))][::-1]
        for i in range(count):
            assert np.array_equal(inorder[i], backward[i]), (limit, i)
        seen.append(inorder)
    assert all(np.array_equal(seen[0][i], insts[i][1]) for i in range(count))
    assert any(not np.array_equal(seen[1][i], seen[2][i]) for i in range(count))
    b.reset()
    assert all(np.array_equal(b.state(i), insts[i][1]) for i in range(count))
