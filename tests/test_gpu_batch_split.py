"""Split batches: plan 6 as (tile, k-mer length, word run) items of every job.

Each case runs the same jobs as plan 6 and as plan 2 (whole 64 x 256 tiles on
the persistent kernel).  Both compute the same 64-bit expressions from the same
exact counts, so every byte is the same.  The shapes sit where the items can go
wrong: one word, one run, runs that do not divide the words, one k-mer length,
single rows and columns, tiles of all three heights, self jobs (upper triangle)
beside query jobs, and a batch whose counts pass the split plan's limit of
32,768 blocks (1,700 tiles x 20 k-mer lengths), which takes the persistent
kernel.
"""
import numpy as np
import pytest

import ppsk_hip as H

pytestmark = pytest.mark.gpu

K5 = [13, 17, 21, 25, 29]


# k-mer lengths, sketchsize64, references, queries per job (0: self job)
@pytest.mark.parametrize("kl,s64,n,queries", [
    (K5, 1, 300, [1, 0, 40]),
    (K5, 7, 257, [17, 0]),
    (K5, 9, 256, [64, 65, 1]),
    ([21], 33, 1, [1, 16]),
    (K5, 156, 700, [113, 0, 31, 300]),
    (list(range(12, 32)), 1, 6200, [4300]),
])
def test_split_equals_whole_tiles(kl, s64, n, queries):
    most = max(queries)
    raw, le, _ = H.synth(n + most, kl, s64, seed=n + s64)
    ref = H.SketchSet(raw[:n], kl, s64, lengths=le[:n])
    qry = [H.SketchSet(raw[n:n + q], kl, s64, lengths=le[n:n + q]) if q else ref for q in queries]
    b = H.Batch([dict(ref=ref, query=q, random_mode=H.RANDOM_EQUAL_BASE if i % 2 else H.RANDOM_NONE,
                      out=("core_acc", "jaccard", "counts")[(i + s64) % 3] if len(kl) > 1 else "jaccard")
                 for i, q in enumerate(qry)])
    try:
        b.run()
        got = {}
        for plan in (2, 6, 6):
            nf, used, _ = b.run(plan)
            assert used == plan
            now = [b.result(x).copy() for x in range(len(qry))]
            if plan in got:
                old_nf, old = got[plan]
                assert np.array_equal(nf, old_nf)
                assert all(np.array_equal(x.view(np.uint8), y.view(np.uint8)) for x, y in zip(now, old))
            got[plan] = (nf, now)
        assert np.array_equal(got[2][0], got[6][0])
        for x, (a, c) in enumerate(zip(got[2][1], got[6][1])):
            assert np.array_equal(a.view(np.uint8), c.view(np.uint8)), (x, kl, s64, n, queries[x])
    finally:
        b.free()
        for q in qry:
            if q is not ref:
                q.free()
        ref.free()
