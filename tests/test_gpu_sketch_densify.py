"""Densification on the GPU against the oracle: sketches with few occupied bins,
whose empty bins take their value through long chains of other empty bins,
from one k-mer to nearly full, at the smallest and the largest sketch sizes and
at sizes that leave some waves of a workgroup without a word.  Words are equal.
"""
import numpy as np
import pytest

import oracle as O
import ppsk_hip as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("s64", [1, 9, 156, 1023])
@pytest.mark.parametrize("windows", [1, 2, 40, 2000])
def test_sparse_bins(s64, windows):
    rng = np.random.default_rng(s64 * 10007 + windows)
    kl = [17, 21]
    samples = [["".join(rng.choice(list("ACGT"), size=windows + 16))],
               ["".join(rng.choice(list("ACGT"), size=windows + 40))],
               ["ACGTN" * 5]]  # no k-mer at all: every bin empty
    raw, mh, dn = H.sketch(samples, kl, s64)
    for x, contigs in enumerate(samples):
        want_mh, want_dn = 0.0, 0
        for i, k in enumerate(kl):
            words, m, d = O.sketch(contigs, k, s64, True)
            assert np.array_equal(raw[x, i], words), (x, k)
            want_mh += m
            want_dn |= int(d != 0)
        assert mh[x] == pytest.approx(want_mh, rel=0, abs=1e-15)
        assert dn[x] == want_dn
