"""Device memory of batches: the counts of a plan that lost the tuning go back, and
a split plan that finds no room leaves nothing behind."""
import numpy as np
import pytest

import ppsk_hip as H

pytestmark = pytest.mark.gpu

KL = list(range(12, 32))


def _free():
    return H.device_init(0)[0]


@pytest.fixture(scope="module")
def sets():
    raw, le, _ = H.synth(8400, KL, 2, seed=3)
    ref = H.SketchSet(raw[:4400], KL, 2, lengths=le[:4400])
    qry = H.SketchSet(raw[4400:], KL, 2, lengths=le[4400:])
    yield ref, qry
    qry.free()
    ref.free()


def _batch(ref, qry, rows):
    return H.Batch([dict(ref=ref, query=qry.prefix(rows), out="counts")])


def test_losing_plan_gives_its_counts_back(sets, monkeypatch):
    # up to 0.7 GiB of counts as plan 6, which whole tiles do without
    ref, qry = sets
    with _batch(ref, qry, 4000) as b:
        b.run(2)  # builds what plan 2 keeps
        before = _free()
        b.run(6)
        assert before - _free() > 300 << 20
        want = b.result(0)
        monkeypatch.setenv("PPSK_BATCH_VARIANT", "2")  # as if plan 2 had been the fastest
        _, used, _ = b.run()
        assert used == 2
        assert before - _free() < 100 << 20
        for plan in (2, 6):
            b.run(plan)
            assert np.array_equal(b.result(0), want)


def test_split_plan_without_room(sets, monkeypatch):
    ref, qry = sets
    with _batch(ref, qry, 1000) as b:
        b.run(2)
        want = b.result(0)
    base = None
    monkeypatch.setenv("PPSK_SCRATCH_BYTES", str(1 << 20))
    for _ in range(4):
        with _batch(ref, qry, 1000) as b:
            _, used, _ = b.run(6)  # on the mixed-shape kernel
            assert used == 6
            assert np.array_equal(b.result(0), want)
        base = base or _free()
    assert base - _free() < 16 << 20
