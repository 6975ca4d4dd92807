"""Serving steps as split passes: every row remainder of a step's tiles.

A step of q queries is laid out in 64-, 32- and 16-row tiles (q = 1 to 130
covers each remainder class and its edges), its counts in launches of whole
column blocks, of at most 8,192 count blocks (53,000 references x 20 k-mer
lengths x 2 tiles take two launches, the last one shorter).  Every step's kNN and
threshold lists equal, bit for bit, those of a server told to split its steps
per (tile, k-mer length):
both compute the same 64-bit expressions from the same counts.
"""
import numpy as np
import pytest

import ppsk_hip as H

pytestmark = pytest.mark.gpu


def _same(a, b):
    assert a["n_fail"] == b["n_fail"]
    for f in ("knn_i", "knn_j", "knn_d", "thr_i", "thr_j", "thr_d"):
        assert np.array_equal(a[f].view(np.uint8), b[f].view(np.uint8)), f


def _both(n, kl, s64, queries, monkeypatch):
    raw, le, _ = H.synth(n + max(queries), kl, s64, seed=n + s64)
    ref = H.SketchSet(raw[:n], kl, s64, lengths=le[:n])
    kw = dict(kNN=5, cutoff=0.05, max_rows=max(queries), n_slots=1,
              random_mode=H.RANDOM_EQUAL_BASE, arena_bytes=2 << 30)
    try:
        res = []
        for forced in (False, True):
            with monkeypatch.context() as m:
                if forced:
                    m.setenv("PPSK_PERSISTENT", "0")
                with H.Server(ref, **kw) as srv:
                    res.append([srv.wait(srv.submit(raw[n:n + q], le[n:n + q])) for q in queries])
        for a, b in zip(*res):
            _same(a, b)
    finally:
        ref.free()


@pytest.mark.parametrize("n,s64", [(300, 9), (256, 1), (257, 156)])
def test_step_rows(n, s64, monkeypatch):
    _both(n, [13, 17, 21, 25, 29], s64,
          [1, 16, 17, 32, 33, 48, 49, 64, 65, 81, 97, 113, 128, 130], monkeypatch)


def test_several_launches(monkeypatch):
    _both(53000, list(range(12, 32)), 1, [3, 20, 40], monkeypatch)
