"""Coded passes cut into several slabs and launches, and full groups.

PPSK_CHUNK_BYTES lowers the counts of a launch, so that a row group's columns are
cut: its rows are coded apart from them, the code buffer serves one launch after
the other and a group's rows are copied to the host after its last slab.  Odd
numbers of k-mer lengths times odd sketches make width tables that are no
multiple of 16 bytes.  Counts are whole numbers and must equal the oracle's.
"""
import numpy as np
import pytest

import oracle as O
import ppsk_hip as H
from test_gpu_split_pass import _alphabets, _pack

pytestmark = pytest.mark.gpu

KLS = {1: [21], 2: [15, 19], 3: [15, 19, 23], 5: [13, 15, 19, 21, 23]}


def _counts(raw, kl, s64, query=None):
    n = len(raw)
    le = np.full(n, 2_000_000, np.uint64)
    kw = {} if query is None else dict(query=query, query_len=le[:1].repeat(len(query)))
    return O.query_db(raw, kl, s64, 14, le, random=O.Random(0, True), jaccard=True,
                      want_counts=True, **kw)[1]


@pytest.mark.parametrize("n,n_k,s64,tiles", [(1300, 3, 5, 22), (1300, 3, 5, 1), (769, 1, 3, 5),
                                             (1537, 5, 1, 60), (800, 2, 4, 13), (1030, 3, 7, 10000)])
def test_self_slabs(monkeypatch, n, n_k, s64, tiles):
    kl = KLS[n_k]
    raw = _pack(_alphabets(n, n_k, s64, 512, n))
    monkeypatch.setenv("PPSK_CODED", "1")
    monkeypatch.setenv("PPSK_CHUNK_BYTES", str(tiles * n_k * 64 * 256 * 2))
    with H.SketchSet(raw, kl, s64) as s:
        c, _, _ = H.dense(s, out="counts")
        dptr, _ = H.dense_device(s, out="counts")
        d = H.copy_to_host(np.empty_like(c), dptr)
        H.device_free(dptr)
    want = _counts(raw, kl, s64)
    assert np.array_equal(c, want)
    assert np.array_equal(d, want)


@pytest.mark.parametrize("q,n,n_k,s64,tiles", [(800, 1000, 3, 5, 30), (800, 1000, 3, 5, 1),
                                               (1537, 257, 1, 3, 20), (65, 2049, 5, 1, 4)])
def test_query_slabs(monkeypatch, q, n, n_k, s64, tiles):
    kl = KLS[n_k]
    raw = _pack(_alphabets(q + n, n_k, s64, min(q, 512), q + n))
    monkeypatch.setenv("PPSK_CODED", "1")
    monkeypatch.setenv("PPSK_CHUNK_BYTES", str(tiles * n_k * 64 * 256 * 2))
    with H.SketchSet(raw[q:], kl, s64) as r, H.SketchSet(raw[:q], kl, s64) as qs:
        c, _, _ = H.dense(r, qs, out="counts")
    assert np.array_equal(c, _counts(raw[q:], kl, s64, query=raw[:q]))


@pytest.mark.parametrize("q,n", [(768, 0), (768, 300), (1536, 130)])
def test_full_group_of_distinct_values(monkeypatch, q, n):
    # 768 rows that all differ at a bin: ranks up to 768, 10 planes; beside bins of
    # few values, columns that hold the same values and others
    kl, s64 = KLS[2], 5
    rng = np.random.default_rng(q + n)
    v = np.zeros((q + n, 2, 64 * s64), np.int64)
    for h in range(2 * s64):
        for kk in range(2):
            a = [768, 1, 767, 3, 600, 513, 16, 512, 64, 700][(h + 3 * kk) % 10]
            for b in range(32 * h, 32 * h + 32):
                letters = rng.permutation(1 << 14)[:a]
                for g in range(0, q, 768):
                    v[g:g + 768, kk, b] = rng.permutation(np.resize(letters, 768))[:min(768, q - g)]
                v[q:, kk, b] = rng.choice(letters, size=n)
                own = rng.random(n) < 0.2
                v[q:, kk, b][own] = rng.integers(0, 1 << 14, size=int(own.sum()))
    raw = _pack(v)
    monkeypatch.setenv("PPSK_CODED", "1")
    with H.SketchSet(raw[q:] if n else raw, kl, s64) as r, H.SketchSet(raw[:q], kl, s64) as qs:
        c, _, _ = H.dense(r, qs if n else None, out="counts")
    want = _counts(raw[q:], kl, s64, query=raw[:q]) if n else _counts(raw, kl, s64)
    assert np.array_equal(c, want)


@pytest.mark.parametrize("n,s64", [(700, 5), (17000, 2)])
def test_full_square_bands(monkeypatch, n, s64):
    # an asymmetric Monte Carlo table: every pair in both orders, in bands of rows
    # from 16,385 samples on; coded and as whole tiles the same bytes
    kl = [13, 17]
    raw, le, _ = H.synth(n, kl, s64, seed=n)
    rng = np.random.default_rng(3)
    cl = rng.integers(0, 3, size=n).astype(np.uint16)
    table = rng.uniform(0, 0.02, size=(2, 3, 3)).astype(np.float32)
    kw = dict(random_mode=H.RANDOM_MC, table=table)
    with H.SketchSet(raw, kl, s64, lengths=le, clusters=cl) as s:
        monkeypatch.setenv("PPSK_CODED", "1")
        got = H.knn(s, 7, **kw)
        monkeypatch.setenv("PPSK_PERSISTENT", "0")
        want = H.knn(s, 7, **kw)
    assert got[3] == want[3]
    for a, b in zip(got[:3], want[:3]):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
