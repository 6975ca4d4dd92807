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


def test_unknown_base_at_every_step():
    # a base that is not A, C, G or T at every position of three blocks of 16
    # steps, and none: blocks with and without unknown bases, before and after
    # the first k, in the same workgroup
    rng = np.random.default_rng(11)
    base = rng.choice(np.frombuffer(b"ACGT", np.uint8), 400)
    samples = [[base.tobytes()]]
    for p in list(range(48)) + [383, 384, 398, 399]:
        seq = base.copy()
        seq[p] = ord("N")
        seq[(p + 200) % 400] = ord("-")
        samples.append([seq.tobytes()])
    raw, _, _ = H.sketch(samples, [3, 13, 31], 1)
    for s, contigs in enumerate(samples):
        for x, k in enumerate([3, 13, 31]):
            assert np.array_equal(raw[s, x], O.sketch(contigs, k, 1, True)[0]), (s, k)


@pytest.mark.parametrize("s64", [1, 16, 156, 1023])
def test_bins_against_oracle(s64):
    # 32-bit bins with the 64-bit way for values next to a bin's end: 120,000
    # windows per k-mer length at the smallest and largest bin counts
    rng = np.random.default_rng(s64)
    seq = rng.choice(np.frombuffer(b"ACGT", np.uint8), 120000).tobytes()
    for use_rc in (True, False):
        raw, mh, _ = H.sketch([[seq]], [15, 27], s64, use_rc=use_rc)
        want = [O.sketch([seq], k, s64, use_rc) for k in (15, 27)]
        for x in range(2):
            assert np.array_equal(raw[0, x], want[x][0]), (s64, use_rc, x)
        assert mh[0] == pytest.approx(want[0][1] + want[1][1], rel=0, abs=1e-15)
