"""Count filter with the rows of hash 1 counted by run of valid k-mers.

A run's k-mers share hash 1, so its events of rows 2 and 3 are one sorted entry
each and an occurrence's count is its place in the run plus the lengths of the
earlier runs on that cell.  Cases: runs of one k-mer and more that start with the
same k-mer (so share both cells), fewer and more occurrences than min_count, one
run, no run, runs cut by unknown bases; and the flat cell that rows 1 and 2 share
(row 1's last index is row 2's first, as in the reference's nested array): k-mers
whose hash lands there (found by search over random 15-mers: bits 27 to 53 of hash
0 all set, bits 0 to 26 of hash 1 all zero) with one side only and with both, where
the job is counted by occurrence.  Words, minhash sums and flags equal the oracle's.
"""
import numpy as np
import pytest

import oracle as O
import ppsk_hip as H

pytestmark = pytest.mark.gpu

ROW1_LAST = ["GCGGTATTACTCTAC", "CCATTTTAGCTCTCT"]
ROW2_FIRST = "GGAGATTGTCGCGAG"


def _check(samples, klist, min_count):
    raw, mh, dn = H.sketch(samples, klist, 16, min_count=min_count)
    for s, contigs in enumerate(samples):
        want_mh, want_dn = 0.0, 0
        for x, k in enumerate(klist):
            us, m, d = O.sketch_filtered(contigs, k, 16, True, min_count, False)
            assert np.array_equal(raw[s, x], us), (s, k, min_count)
            want_mh += m
            want_dn |= int(d != 0)
        assert mh[s] == want_mh, s
        assert dn[s] == want_dn, s


def _reads(seed, copies):
    rng = np.random.default_rng(seed)
    out = []
    for n, c in copies:
        base = rng.choice(list("ACGT"), size=n)
        for x in range(c):  # same start, lengths n, n - 1, ... and back
            out.append("".join(base[: max(1, n - x % 5)]))
    order = rng.permutation(len(out))
    return [out[i] for i in order]


@pytest.mark.parametrize("min_count", [1, 2, 3, 6, 40, 255])
def test_runs_that_share_cells(min_count):
    samples = [_reads(1, [(15, 9), (16, 4), (20, 7), (40, 60), (90, 3)]),
               _reads(2, [(300, 1)]),
               _reads(3, [(14, 3)]),
               _reads(4, [(150, 2)] * 200 + [(17, 300)]),
               [r[:30] + "N" + r[30:] for r in _reads(5, [(120, 3)] * 60)]]
    _check(samples, [15, 17], min_count)


@pytest.mark.parametrize("min_count", [2, 3, 5])
def test_cell_between_rows(min_count):
    rng = np.random.default_rng(8)

    def around(mid, first):
        tail = "".join(rng.choice(list("ACGT"), size=60))
        return (first + tail[:30] + mid + tail[30:]) if first else (tail[:30] + mid + tail[30:])

    plain = _reads(9, [(150, 4)] * 50)
    occurrence = [around(ROW1_LAST[x % 2], "") for x in range(6)]
    run = [around("", ROW2_FIRST) for _ in range(6)]
    both = [around(ROW1_LAST[x % 2], ROW2_FIRST) for x in range(6)]
    _check([plain, plain + occurrence * 2, plain + run * 2, occurrence + run + plain,
            run + occurrence + plain + both, both[:1]], [15], min_count)
