"""Mid-pass cancellation and progress on the routes that calls take by default.

Split and coded passes, also those of a few milliseconds, look for a cancellation
between their items, mirror their progress to the host while they run and leave no
state behind.  A short pass may end before the request reaches it, so the request
is made again in up to 40 calls; one that stops early is enough.
"""
import threading

import numpy as np
import pytest

import ppsk_hip as H
from helpers import KLIST8, synth
from test_gpu_cancel import N_BIG, S64, _check_small_against_oracle, _run_and_cancel

pytestmark = pytest.mark.gpu


def _cancel_short(call):
    """(progress of the call that stopped early, calls made) or (None, calls)."""
    for calls in range(1, 41):
        H.cancel_reset(0)
        box = {}

        def target():
            try:
                call()
            except H.PpskError as e:
                box["err"] = e

        th = threading.Thread(target=target)
        th.start()
        while th.is_alive():
            st = H.progress(0)
            if st["running"] and st["done"] > 0:
                H.cancel(0)
                break
        th.join()
        final = H.progress(0)
        H.cancel_reset(0)
        if "err" in box:
            assert box["err"].code == H.ERR_CANCELLED
            if final["done"] < final["total"]:
                return final, calls
    return None, calls


def test_cancel_large_pass_default_route():
    raw, le, _ = H.synth(N_BIG, KLIST8, S64, seed=31)
    with H.SketchSet(raw, KLIST8, S64, lengths=le) as big:
        del raw
        dptr = H.device_alloc(N_BIG * (N_BIG - 1) // 2 * 8)
        try:
            err, seen, final = _run_and_cancel(lambda: H.dense_device(big, dptr=dptr))
        finally:
            H.device_free(dptr)
    assert seen is not None, "the pass ended before any progress was seen"
    assert err is not None and err.code == H.ERR_CANCELLED
    assert 0 < final["done"] < final["total"]
    _check_small_against_oracle()


@pytest.mark.parametrize("coded", ["1", "0"])
def test_cancel_short_pass(monkeypatch, coded):
    raw, le, _ = synth(3000)  # 4.5 ms coded, 5 ms on the planes
    with H.SketchSet(raw, KLIST8, S64, lengths=le) as s:
        monkeypatch.setenv("PPSK_CODED", coded)
        want, nf = H.dense_device(s)
        try:
            final, _ = _cancel_short(lambda: H.dense_device(s, dptr=want))
            assert final is not None
            assert not final["running"]
            # whole again
            H.dense_device(s, dptr=want)
            st = H.progress(0)
            assert st["done"] == st["total"] > 0
            a = H.copy_to_host(np.empty((3000 * 2999 // 2, 2), np.float32), want)
            monkeypatch.setenv("PPSK_PERSISTENT", "0")
            assert np.array_equal(a, H.dense(s)[0])
        finally:
            H.device_free(want)


def test_cancel_split_batch():
    raw, le, _ = synth(3000)
    with H.SketchSet(raw[:2500], KLIST8, S64) as r, H.SketchSet(raw[2500:], KLIST8, S64) as q:
        with H.Batch([dict(ref=r, query=q), dict(ref=r, query=r), dict(ref=r, query=q.prefix(30))]) as b:
            b.run(2)
            want = [b.result(x) for x in range(3)]
            b.run(6)
            final, _ = _cancel_short(lambda: b.run(6))
            assert final is not None
            b.run(6)
            for x in range(3):
                assert np.array_equal(b.result(x).view(np.uint8), want[x].view(np.uint8))
