"""Split passes: (tile, k-mer length, word run) items and the separate output
kernel, at the edges of the tile heights (16, 32, 64 rows), of the 256-column
tiles and of the word runs (sketches of fewer words than a stage, runs that do
not divide the sketch), against the oracle: counts bit-exact, core/accessory
within the 1e-6 of the other parity tests.
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
