"""Split passes: (tile, k-mer length, word run) items and the separate output
kernel, at the edges of the tile heights (16, 32, 64 rows), of the 256-column
tiles and of the word runs (sketches of fewer words than a stage, runs that do
not divide the sketch), against the oracle: counts bit-exact, core/accessory
within the 1e-6 of the other parity tests.

Coded passes (a row group's values as ranks): every width of the codes, from
bins where all rows agree to 512 rows that all differ, in runs next to each
other; columns holding values that no row holds; groups, tiles and blocks with
remainders; unrelated samples.  Counts are whole numbers and must be equal.
"""
import numpy as np
import pytest

import oracle as O
import ppsk_hip as H
from helpers import synth

pytestmark = pytest.mark.gpu

KL = (15, 19, 23)


@pytest.mark.parametrize("q,n,s64", [(1, 255, 156), (16, 257, 3), (17, 300, 1), (33, 100, 5),
                                     (49, 513, 7), (65, 1, 2), (113, 260, 313)])
def test_query_edges(q, n, s64):
    raw, le, _ = synth(q + n, KL, s64)
    with H.SketchSet(raw[q:], KL, s64, lengths=le[q:]) as r, \
            H.SketchSet(raw[:q], KL, s64, lengths=le[:q]) as qs:
        c, _, _ = H.dense(r, qs, out="counts")
        d, nf, _ = H.dense(r, qs, random_mode=H.RANDOM_EQUAL_BASE)
    want, want_c, wnf, _ = O.query_db(raw[q:], KL, s64, 14, le[q:], query=raw[:q],
                                      query_len=le[:q], random=O.Random(1, True),
                                      want_counts=True)
    assert np.array_equal(c, want_c)
    assert nf == wnf
    assert np.abs(d - want).max() <= 1e-6


@pytest.mark.parametrize("n,s64", [(2, 4), (17, 156), (64, 9), (257, 6), (321, 30)])
def test_self_edges(n, s64):
    raw, le, _ = synth(n, KL, s64)
    with H.SketchSet(raw, KL, s64, lengths=le) as s:
        c, _, _ = H.dense(s, out="counts")
        j, _, _ = H.dense(s, out="jaccard", random_mode=H.RANDOM_EQUAL_BASE)
    want_j, want_c, _, _ = O.query_db(raw, KL, s64, 14, le, random=O.Random(1, True),
                                      jaccard=True, want_counts=True)
    assert np.array_equal(c, want_c)
    assert np.array_equal(j.view(np.uint32), want_j.view(np.uint32))


def _pack(v):
    """Bin values [n][n_k][64 s64] -> words [n][n_k][s64 * 14]."""
    n, n_k, bins = v.shape
    x = v.reshape(n, n_k, bins // 64, 64).astype(np.uint64)
    out = np.zeros((n, n_k, bins // 64, 14), np.uint64)
    for b in range(14):
        out[..., b] = (((x >> np.uint64(b)) & np.uint64(1)) << np.arange(64, dtype=np.uint64)).sum(
            -1, dtype=np.uint64)
    return out.reshape(n, n_k, -1)


def _alphabets(n, n_k, s64, distinct_rows, seed):
    """Values whose number of distinct ones changes from each run of 32 bins
    to the next (1 .. 512), spread over the 14 bits; the first distinct_rows
    samples all differ in some runs, the others also draw values of their own."""
    rng = np.random.default_rng(seed)
    sizes = [1, 7, 8, 15, 16, 40, 63, 64, 127, 128, 255, 256, 300, 511, 512, 16384]
    v = np.zeros((n, n_k, 64 * s64), np.int64)
    for h in range(2 * s64):
        for kk in range(n_k):
            a = sizes[(h * 5 + kk) % len(sizes)]
            letters = rng.permutation(1 << 14)[:a]
            cells = letters[rng.integers(0, a, size=(n, 32))]
            if a >= 256:  # every one of the first rows another value
                m = min(a, distinct_rows)
                cells[:m] = np.stack([rng.permutation(letters)[:m] for _ in range(32)], 1)
            own = rng.random((n, 32)) < 0.1
            own[:distinct_rows] = False
            cells[own] = rng.integers(0, 1 << 14, size=int(own.sum()))
            v[:, kk, 32 * h:32 * h + 32] = cells
    return v


@pytest.mark.parametrize("n,s64,rows", [(512, 17, 512), (601, 8, 320), (1100, 3, 384),
                                        (300, 1, 256), (64, 5, 64)])
def test_coded_self(monkeypatch, n, s64, rows):
    monkeypatch.setenv("PPSK_CODED", "1")
    kl = [15, 19, 23]
    raw = _pack(_alphabets(n, 3, s64, rows, n))
    with H.SketchSet(raw, kl, s64) as s:
        c, _, _ = H.dense(s, out="counts")
        monkeypatch.setenv("PPSK_CODED", "0")
        plain, _, _ = H.dense(s, out="counts")
    want = O.query_db(raw, kl, s64, 14, np.full(n, 2_000_000, np.uint64), random=O.Random(0, True),
                      jaccard=True, want_counts=True)[1]
    assert np.array_equal(plain, want)
    assert np.array_equal(c, want)


@pytest.mark.parametrize("q,n,s64", [(1, 300, 4), (17, 256, 9), (449, 513, 6), (520, 1000, 3),
                                     (64, 130, 157)])
def test_coded_query(monkeypatch, q, n, s64):
    monkeypatch.setenv("PPSK_CODED", "1")
    kl = [15, 19]
    raw = _pack(_alphabets(q + n, 2, s64, min(q, 512), q + n))
    le = np.full(q + n, 2_000_000, np.uint64)
    with H.SketchSet(raw[q:], kl, s64, lengths=le[q:]) as r, \
            H.SketchSet(raw[:q], kl, s64, lengths=le[:q]) as qs:
        c, _, _ = H.dense(r, qs, out="counts")
        with r.prefix(max(1, n - 100)) as part:
            cp, _, _ = H.dense(part, qs, out="counts")
    want = O.query_db(raw[q:], kl, s64, 14, le[q:], query=raw[:q], query_len=le[:q],
                      random=O.Random(0, True), jaccard=True, want_counts=True)[1]
    assert np.array_equal(c, want)
    assert np.array_equal(cp.reshape(q, -1, 2), want.reshape(q, n, 2)[:, :max(1, n - 100)])


def test_coded_default_route_and_word_runs(monkeypatch):
    # 900 tree samples take the coded route by themselves, words cut into runs;
    # the planes route gives the same bytes
    raw, le, _ = synth(900)
    with H.SketchSet(raw, list(range(15, 30, 2)), 156, lengths=le) as s:
        d, nf, _ = H.dense(s, random_mode=H.RANDOM_EQUAL_BASE)
        monkeypatch.setenv("PPSK_CODED", "0")
        d0, nf0, _ = H.dense(s, random_mode=H.RANDOM_EQUAL_BASE)
    assert nf == nf0 == 0
    assert np.array_equal(d.view(np.uint32), d0.view(np.uint32))
