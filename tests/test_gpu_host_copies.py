"""Copies between host memory and the device through page-locked blocks.

Blocks are 2 MiB, one thread below 4 MiB and up to four from there on: the sizes
are the edges of a block, of the thread count and of several turns of every
block, at unaligned host addresses.  Exact comparison of bytes.
"""
import threading

import numpy as np
import pytest

import ppsk_hip as H

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.fixture(scope="module")
def wide():
    rng = np.random.default_rng(1)
    raw = rng.integers(0, 1 << 63, size=(1150000, 1, 14), dtype=np.uint64)
    ref = H.SketchSet(raw, [17], 1)
    qry = H.SketchSet(raw[1000:1016], [17], 1)
    yield ref, qry
    qry.free()
    ref.free()


# 2 bytes per pair
@pytest.mark.parametrize("q,n", [(1, 1), (1, 3), (1, MB - 1), (1, MB), (1, MB + 1), (2, MB - 1),
                                 (2, MB), (2, MB + 1), (16, 600001), (16, 1150000)])
def test_copy_to_host(wide, q, n):
    ref, qry = wide
    r, s = ref.prefix(n), qry.prefix(q)
    got = H.dense(r, s, out="counts")[0]
    dptr, _ = H.dense_device(r, s, out="counts")
    want = np.zeros_like(got)
    H.copy_to_host(want, dptr)
    H.device_free(dptr)
    assert np.array_equal(got, want)
    if n > 1016:
        assert (got.reshape(q, n)[np.arange(q), 1000 + np.arange(q)] == 64).all()
    r.free()
    s.free()


@pytest.mark.parametrize("n", [1, 40, 300, 333, 700])
def test_upload_in_one_and_in_parts(n):
    # 140 KB a sample: up to three chunks of 32 MiB; the same set uploaded in
    # one call and sample by sample gives the same counts
    kl = [13, 17, 21, 25, 29, 31, 33, 35]
    raw, _, _ = H.synth(max(n, 2), kl, 156, seed=n)
    raw = raw[:n]
    one = H.SketchSet(raw, kl, 156)
    parts = H.SketchSet(raw, kl, 156)
    try:
        for x in range(n):
            H.lib().ppsk_set_upload(parts.handle, x, 1, H._ptr(np.ascontiguousarray(raw[x])))
        q = H.SketchSet(raw[: max(1, n // 7)][::-1].copy(), kl, 156)
        a = H.dense(one, q, out="counts")[0]
        b = H.dense(parts, q, out="counts")[0]
        q.free()
        assert np.array_equal(a, b)
        # the queries are the first samples: each matches itself in every bin
        m = max(1, n // 7)
        own = a.reshape(m, n, len(kl))[np.arange(m), m - 1 - np.arange(m)]
        assert (own == 156 * 64).all()
    finally:
        one.free()
        parts.free()


def test_contigs_where_they_are():
    # long contigs are gathered from where they lie, short ones joined: the same
    # samples cut into contigs at both sides of 4,096 bytes, empty ones among them
    rng = np.random.default_rng(5)
    big = [bytes(rng.choice(list(b"ACGT"), size=s).astype(np.uint8)) for s in (5 * MB, 0, 4096, 3 * MB + 1)]
    a = H.sketch([big, big[2:]], [13, 17, 21], 64)
    pad = [b""] * 2000  # 2,008 contigs, mean length below 4,096
    b = H.sketch([big + pad, big[2:] + pad + pad], [13, 17, 21], 64)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


def test_set_memory_is_cleared_and_shared_safely():
    # sets created and freed from several threads: memory of a freed set serves
    # the next one, whose samples beyond an upload are zero again
    kl = [13, 17, 21]
    raw, _, _ = H.synth(64, kl, 16, seed=3)
    want = H.dense(H.SketchSet(raw, kl, 16), None, out="counts")[0]
    bad = []

    def work():
        for _ in range(20):
            s = H.SketchSet(raw, kl, 16)
            got = H.dense(s, None, out="counts")[0]
            s.free()
            if not np.array_equal(got, want):
                bad.append(1)

    t = [threading.Thread(target=work) for _ in range(4)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    assert not bad
