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
