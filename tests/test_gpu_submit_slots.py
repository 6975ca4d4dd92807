"""ppsk_server_submit copies the queries and never waits for the GPU, whatever the
number of slots, and ppsk_server_free waits for a submit that began before it."""
import threading
import time

import numpy as np
import pytest

import ppsk_hip as H
from helpers import KLIST8

pytestmark = pytest.mark.gpu

S64 = 156


def test_submit_beside_many_slots():
    # 8 steps of 128 queries x 30,000 references (about 4 ms each) in flight feed the
    # 4 hardware queues of the process
    n = 30000
    raw, le, _ = H.synth(n + 128, KLIST8, S64, seed=21, dcore_max=0.15)
    ref = H.SketchSet(raw[:n], KLIST8, S64, lengths=le[:n])
    q, ql = raw[n:].copy(), le[n:].copy()
    del raw
    worst = 0.0
    with H.Server(ref, kNN=10, cutoff=0.05, random_mode=H.RANDOM_EQUAL_BASE, n_slots=8,
                  arena_bytes=16 << 30) as srv:
        first = srv.wait(srv.submit(q[:1], ql[:1]))
        big = [srv.submit(q, ql) for _ in range(48)]
        small = []
        for _ in range(40):
            t = time.perf_counter()
            small.append(srv.submit(q[:1], ql[:1]))
            worst = max(worst, time.perf_counter() - t)
            time.sleep(0.002)
        for t in big:
            srv.wait(t)
        for t in small:
            r = srv.wait(t)
            assert np.array_equal(r["knn_j"], first["knn_j"])
            assert np.array_equal(r["thr_j"], first["thr_j"])
    ref.free()
    print(f"longest submit of one query {worst * 1e3:.2f} ms")
    assert worst < 0.005


def test_free_waits_for_a_submit():
    # a submit of 800,000 queries computes for about 0.1 s before it queues them
    kl = [13, 17]
    raw, le, _ = H.synth(2, kl, 1, seed=3)
    ref = H.SketchSet(raw[:1], kl, 1, lengths=le[:1])
    many, ml = np.repeat(raw[1:], 800_000, 0), np.repeat(le[1:], 800_000)
    srv = H.Server(ref, kNN=1, cutoff=0.0, random_mode=H.RANDOM_EQUAL_BASE, max_rows=250_000, n_slots=1,
                   arena_bytes=1 << 30)
    srv.wait(srv.submit(many[:10], ml[:10]))
    box = {}

    def target():
        t = time.perf_counter()
        try:
            srv.submit(many, ml)
            box["rc"] = H.OK
        except H.PpskError as e:
            box["rc"] = e.code
        box["s"] = time.perf_counter() - t

    th = threading.Thread(target=target)
    th.start()
    time.sleep(0.02)
    srv.free()
    th.join()
    assert box["rc"] in (H.OK, H.ERR_STATE)
    ref.free()
