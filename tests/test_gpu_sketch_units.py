"""Work units of a sketching call, written on the device from running counts.

Contig lengths at the edges of a window (0, k - 1, k, k + 1), of the shortest unit
(64 windows) and of the longest (1,024 windows, the read sets' unit), in several
samples (one of them a single contig, one without a window at the longest k) and
in both orders, against the oracle: sketch words, minhash sums and densified flags
are the same.
"""
import numpy as np
import pytest

import oracle as O
import ppsk_hip as H

pytestmark = pytest.mark.gpu

KL = [13, 21, 31]
LENGTHS = [0, 12, 13, 14, 20, 21, 22, 30, 31, 32, 76, 77, 94, 95, 416, 447, 1035, 1036, 1037,
           1044, 1054, 1055, 2060, 2061, 3105, 0]


def _samples():
    rng = np.random.default_rng(9)
    base = rng.choice(np.frombuffer(b"ACGT", np.uint8), 40000)

    def cut(lengths):
        at = rng.integers(0, len(base) - 4000, len(lengths))
        return [base[a:a + n].tobytes() for a, n in zip(at, lengths)]

    return [cut(LENGTHS), cut(LENGTHS[::-1]), [base.tobytes()], cut([25, 0, 30]), cut([3000] * 40)]


@pytest.mark.parametrize("min_count,exact", [(0, False), (1, False), (2, False), (2, True)])
def test_units_against_oracle(min_count, exact):
    samples = _samples()
    raw, mh, dn = H.sketch(samples, KL, 16, min_count=min_count, exact=exact)
    for s, contigs in enumerate(samples):
        want_mh, want_dn = 0.0, 0
        for x, k in enumerate(KL):
            if min_count:
                us, m, d = O.sketch_filtered(contigs, k, 16, True, min_count=min_count, exact=exact)
            else:
                us, m, d = O.sketch(contigs, k, 16, True)
            assert np.array_equal(raw[s, x], us), (s, k)
            want_mh += m
            want_dn |= int(d != 0)
        assert mh[s] == pytest.approx(want_mh, rel=0, abs=1e-15), s
        assert dn[s] == want_dn, s
