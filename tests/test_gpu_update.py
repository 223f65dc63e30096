"""The sorted update at the edges of its label sort's two scans: one block's
(histograms of up to 20,480 counts; with more of them in up to 512K rows, ranges
of more rows while 96 remain) and three launches."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [
    (300, 65), (26_112, 200), (26_113, 200), (40_001, 213), (40_001, 214), (20_480, 256), (20_481, 256),
    (5_000, 1024), (5_400, 1025), (525_000, 70),
])
def test_sums_at_the_scans_edges(n, k):
    from skmetal_amd import _bridge

    rng = np.random.default_rng(n + k)
    d = 20
    C = (8.0 * rng.standard_normal((k, d))).astype(np.float32)
    want = rng.integers(0, k, n)
    want[:k] = rng.permutation(k) if n >= k else want[:k]
    X = (C[want] + 0.1 * rng.standard_normal((n, d))).astype(np.float32)
    with _bridge.LloydHandle(n, d, k) as h:
        h.load(X, center=False)
        h.set_centers(C)
        h.iterate(1)
        lab, new = h.labels(), h.centers()
    np.testing.assert_array_equal(lab, want)  # (centres far apart)
    cnt = np.bincount(want, minlength=k)
    for c in range(d):
        x = X[:, c].astype(np.float64)
        mean = np.bincount(want, weights=x, minlength=k) / cnt
        size = np.bincount(want, weights=np.abs(x), minlength=k) / cnt
        # fp32 chains over a chunk of at most 512 rows, fp64 across them, an fp32 result
        assert np.all(np.abs(new[:, c] - mean) <= np.minimum(cnt, 512) * 2.0**-24 * size + 2.0**-24 * np.abs(mean))
