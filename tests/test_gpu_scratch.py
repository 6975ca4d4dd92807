"""Calls where the device has room for only part of the scratch that they would take.

PPSK_SCRATCH_BYTES refuses workspaces past a limit as a full device does.  A
self pass of 3,000 samples takes about 0.8 GiB of codes and 0.2 GiB of counts:
below that it runs with fewer codes at a time, then on the planes, then as
whole tiles, which took 80 MiB before passes were split.  Every route computes the
same 64-bit expressions from the same exact counts, so every byte is the same.
"""
import os
import subprocess
import sys

import numpy as np
import pytest

import ppsk_hip as H
from helpers import KLIST8, synth

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.fixture(scope="module")
def sets():
    raw, le, _ = synth(3000)
    s = H.SketchSet(raw, KLIST8, 156, lengths=le)
    q = H.SketchSet(raw[:300], KLIST8, 156, lengths=le[:300])
    kw = dict(random_mode=H.RANDOM_EQUAL_BASE)
    with pytest.MonkeyPatch.context() as m:
        m.setenv("PPSK_PERSISTENT", "0")  # whole tiles: a split pass's scratch is not there yet
        full = (H.dense(s, **kw)[0], H.dense(s, q, **kw)[0], H.knn(s, 10, **kw), H.threshold(s, 0.01, **kw))
    yield s, q, full
    q.free()
    s.free()


def _same(a, b):
    return np.array_equal(np.asarray(a).view(np.uint8), np.asarray(b).view(np.uint8))


@pytest.mark.parametrize("limit", [100, 150, 200, 300, 400, 512, 700, 900, 1100])
def test_less_scratch_same_bytes(sets, monkeypatch, limit):
    s, q, (dense, query, knn, thr) = sets
    kw = dict(random_mode=H.RANDOM_EQUAL_BASE)
    monkeypatch.setenv("PPSK_SCRATCH_BYTES", str(limit * MB))
    assert _same(H.dense(s, **kw)[0], dense)
    st = H.progress(0)
    assert st["done"] == st["total"] > 0
    assert _same(H.dense(s, q, **kw)[0], query)
    assert all(_same(a, b) for a, b in zip(H.knn(s, 10, **kw)[:3], knn[:3]))
    assert all(_same(a, b) for a, b in zip(H.threshold(s, 0.01, **kw)[:3], thr[:3]))


@pytest.mark.parametrize("limit", [60, 100])
def test_whole_tiles_on_the_persistent_kernel(monkeypatch, limit):
    # 1,046 tiles: two per resident workgroup, so that the last resort is the
    # persistent kernel (50 MiB) and not one workgroup per (tile, k-mer length)
    kl = [15, 21]
    raw, le, _ = H.synth(5800, kl, 20, seed=4)
    with H.SketchSet(raw, kl, 20, lengths=le) as s:
        kw = dict(random_mode=H.RANDOM_EQUAL_BASE, out="jaccard")
        with monkeypatch.context() as m:
            m.setenv("PPSK_PERSISTENT", "0")
            want = H.dense(s, **kw)[0]
        monkeypatch.setenv("PPSK_SCRATCH_BYTES", str(limit * MB))
        assert _same(H.dense(s, **kw)[0], want)
        st = H.progress(0)
        assert st["done"] == st["total"] > 0


def test_no_scratch_is_an_error(sets, monkeypatch):
    s, q, (dense, _, _, _) = sets
    kw = dict(random_mode=H.RANDOM_EQUAL_BASE)
    monkeypatch.setenv("PPSK_SCRATCH_BYTES", "100000")
    for call in (lambda: H.dense(s, **kw), lambda: H.dense(s, q, **kw), lambda: H.knn(s, 10, **kw)):
        with pytest.raises(H.PpskError) as e:
            call()
        assert e.value.code == H.ERR_MEMORY
    monkeypatch.delenv("PPSK_SCRATCH_BYTES")
    assert _same(H.dense(s, **kw)[0], dense)


def test_codes_go_back_with_the_last_set(sets):
    # 4,608 samples: about 1.7 GiB of codes.  With the module's sets alive they stay
    # for the next pass; a program that has freed its sets gets them back.
    code = """if True:
        import ppsk_hip as H
        kl = list(range(15, 30, 2))
        raw, _, _ = H.synth(4608, kl, 156, seed=2)
        for _ in range(2):
            s = H.SketchSet(raw, kl, 156)
            d, _ = H.dense_device(s)
            alive = H.device_init(0)[0]
            H.device_free(d)
            s.free()
            print(H.device_init(0)[0] - alive)
    """
    out = subprocess.run([sys.executable, "-c", code], check=True, capture_output=True, text=True,
                         env={**os.environ, "PYTHONPATH": os.pathsep.join(sys.path)}, timeout=100).stdout
    stripes = 8 * 36 * 156 * 28 * 128 * 4
    for freed in map(int, out.split()):
        assert freed > stripes + 4608 * 4607 // 2 * 8 + (1 << 30)
