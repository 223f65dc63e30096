"""Relocation that empties the clusters it takes rows from: a cluster of one far
row gives it away, stays empty, and takes the heaviest cluster's centre
(sklearn/cluster/_k_means_common.pyx:167-211, :274-295).  The next E-step needs
that centre's own norm."""

from __future__ import annotations

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _problem(n, d, k, seed):
    """k - 6 blobs of rows, three clusters of one row away from its centre, three
    centres that tie with the first ones and stay empty."""
    rng = np.random.default_rng(seed)
    C = 4.0 * rng.standard_normal((k, d))
    lab = rng.integers(0, k - 6, n)
    lab[: k - 6] = np.arange(k - 6)
    X = C[lab] + 0.1 * rng.standard_normal((n, d))
    for i in range(3):
        X[n - 1 - i] = C[k - 6 + i] + 0.5 + 0.1 * i
    C[k - 3:] = C[:3]
    return X.astype(np.float32), C.astype(np.float32)


# the fused steps (fp32, split), the generic one with the sorted update for short
# and long rows, screened or not
SHAPES = [(4000, 8, 12), (4000, 12, 40), (4000, 32, 20), (9000, 100, 60), (4000, 40, 90), (6000, 64, 200),
          (5000, 150, 150), (3000, 600, 140)]


@pytest.mark.parametrize("n,d,k,screen", [(*s, "0") for s in SHAPES] + [(*s, "1") for s in SHAPES if s[2] > 128])
def test_emptied_donors(monkeypatch, n, d, k, screen):
    from skmetal_amd import _bridge

    monkeypatch.setenv("SKMETAL_HIP_SCREEN", screen)
    X, C = _problem(n, d, k, n + d)
    Xc = X - X.mean(axis=0)
    for steps in (1, 2, 3):
        with _bridge.LloydHandle(n, d, k) as h:
            h.load(Xc, center=False)
            h.set_centers(C - X.mean(axis=0))
            h.run(steps, 0.0, strict=False)  # ends in an E-step of its own
            lab, cen = h.labels(), h.centers()
        ref = oracle.lloyd(Xc, C - X.mean(axis=0), steps)
        if steps == 1:  # the case is the one meant: clusters without a row after the relocation
            first = oracle.assign(Xc, C - X.mean(axis=0))
            cnt = np.bincount(first, minlength=k)
            assert (cnt == 0).sum() == 3 and (cnt == 1).sum() >= 3
        np.testing.assert_allclose(cen, ref["centers"], rtol=1e-4, atol=1e-3)
        np.testing.assert_array_equal(lab, oracle.assign(Xc, cen))
