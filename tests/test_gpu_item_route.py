"""Passes and serving steps of more than two tiles per resident workgroup, which run
as split items and not as whole tiles of the persistent kernel, and the heights
of the last rows' tiles on both sides of their rule (64 pairs of a 64-row tile and
a k-mer length; more than 32 or 48 rows left).  Every byte is the same as with the
persistent kernel or one workgroup per (tile, k-mer length).
"""
import numpy as np
import pytest

import ppsk_hip as H
from helpers import mc_table

pytestmark = pytest.mark.gpu

KL = [15, 21]


def _bytes(a):
    return np.ascontiguousarray(a).view(np.uint8)


@pytest.fixture(scope="module")
def wide():
    n = 135_000
    raw, le, _ = H.synth(n + 513, KL, 1, seed=9)
    cl = (np.arange(n + 513) % 3).astype(np.uint16)
    ref = H.SketchSet(raw[:n], KL, 1, lengths=le[:n], clusters=cl[:n])
    yield ref, raw[n:], le[n:], cl[n:]
    ref.free()


@pytest.mark.parametrize("q,out,mode", [(65, "core_acc", H.RANDOM_EQUAL_BASE), (80, "jaccard", H.RANDOM_NONE),
                                        (97, "counts", H.RANDOM_NONE), (129, "jaccard", H.RANDOM_MC)])
def test_query_over_many_columns(wide, monkeypatch, q, out, mode):
    ref, raw, le, cl = wide
    table = mc_table(KL)[0] if mode == H.RANDOM_MC else None
    with H.SketchSet(raw[:q], KL, 1, lengths=le[:q], clusters=cl[:q]) as s:
        kw = dict(out=out, random_mode=mode, table=table)
        monkeypatch.setenv("PPSK_CODED", "0")
        got = H.dense(ref, s, **kw)
        monkeypatch.setenv("PPSK_PERSISTENT", "1")
        want = H.dense(ref, s, **kw)
    assert got[1:] == want[1:]
    assert np.array_equal(_bytes(got[0]), _bytes(want[0]))


@pytest.mark.parametrize("rows", [1, 16, 17, 32, 33, 48, 49, 64, 96, 97, 112, 113])
@pytest.mark.parametrize("n", [200, 4000, 9000])  # 2 to 64 pairs and more
def test_heights_of_the_last_rows(monkeypatch, rows, n):
    raw, le, _ = H.synth(n + rows, KL, 3, seed=n)
    with H.SketchSet(raw[:n], KL, 3, lengths=le[:n]) as ref, \
            H.SketchSet(raw[n:], KL, 3, lengths=le[n:]) as s:
        for coded in ("0", "1"):
            monkeypatch.setenv("PPSK_CODED", coded)
            got = H.dense(ref, s, out="counts")[0]
            monkeypatch.setenv("PPSK_PERSISTENT", "0")
            assert np.array_equal(got, H.dense(ref, s, out="counts")[0])
            monkeypatch.delenv("PPSK_PERSISTENT")


@pytest.mark.parametrize("rows", [40, 70, 97, 128])
def test_serving_steps(wide, monkeypatch, rows):
    ref, raw, le, cl = wide
    kw = dict(kNN=5, cutoff=0.01, random_mode=H.RANDOM_EQUAL_BASE, max_rows=128, n_slots=1,
              arena_bytes=2 << 30)
    with H.Server(ref, **kw) as srv:
        got = srv.wait(srv.submit(raw[:rows].copy(), le[:rows]))
    monkeypatch.setenv("PPSK_PERSISTENT", "1")  # 70 rows: 28 tiles past two rounds go to the tail
    with H.Server(ref, **kw) as srv:
        want = srv.wait(srv.submit(raw[:rows].copy(), le[:rows]))
    for k in ("knn_i", "knn_j", "knn_d", "thr_i", "thr_j", "thr_d"):
        assert np.array_equal(_bytes(got[k]), _bytes(want[k])), k
    assert got["n_fail"] == want["n_fail"]
