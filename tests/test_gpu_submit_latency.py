"""A server's submit does not wait for another call's kernels.

Copies between ordinary host memory and a device share a few page-locked blocks
and their lock.  While a long pass runs, other threads upload sketches (whose
stripes are queued behind the pass) and set lengths; a submit of one query takes
a copy of 140 KB and must not take a large part of the pass.
"""
import threading
import time

import numpy as np
import pytest

import ppsk_hip as H
from helpers import KLIST8

pytestmark = pytest.mark.gpu

S64 = 156
N_BIG = 24576  # about 0.25 s


@pytest.mark.parametrize("other", ["upload", "meta"])
def test_submit_beside_a_long_pass(other):
    raw, le, _ = H.synth(N_BIG, KLIST8, S64, seed=31)
    big = H.SketchSet(raw, KLIST8, S64, lengths=le)
    some = H.SketchSet(raw[:700], KLIST8, S64, lengths=le[:700])  # 98 MB: four chunks of 32 MiB
    ref = H.SketchSet(raw[:64], KLIST8, S64)
    part, one = raw[:700].copy(), raw[:1].copy()
    del raw
    out = H.device_alloc(N_BIG * (N_BIG - 1) // 2 * 8)
    worst = 0.0
    try:
        with H.Server(ref, kNN=1, arena_bytes=1 << 30) as srv:
            srv.wait(srv.submit(one))
            H.dense_device(big, dptr=out)
            t0 = time.perf_counter()
            H.dense_device(big, dptr=out)
            alone = time.perf_counter() - t0
            done = threading.Event()

            def run_pass():
                H.dense_device(big, dptr=out)
                done.set()

            def run_other():
                if other == "upload":
                    H.lib().ppsk_set_upload(some.handle, 0, 700, H._ptr(part))
                else:
                    H.lib().ppsk_set_meta(some.handle, H._ptr(le[:700].copy()), 1, None)

            a, b = threading.Thread(target=run_pass), threading.Thread(target=run_other)
            a.start()
            time.sleep(0.03 * alone / 0.25)
            b.start()
            time.sleep(0.03 * alone / 0.25)
            tickets, during = [], 0
            while not done.is_set():
                t0 = time.perf_counter()
                tickets.append(srv.submit(one))
                worst = max(worst, time.perf_counter() - t0)
                during += not done.is_set()
                time.sleep(0.002)
            a.join()
            b.join()
            for t in tickets:
                srv.wait(t)
        print(f"pass {alone * 1e3:.1f} ms, {during} submits beside it, longest {worst * 1e3:.2f} ms")
        assert during >= 5
        assert worst < 0.3 * alone
    finally:
        H.device_free(out)
        for s in (big, some, ref):
            s.free()
