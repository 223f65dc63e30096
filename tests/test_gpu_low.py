"""k_fused_low (rows of at most 16 floats): one Lloyd step against an fp64 step
from the same centres, at the edges of its tiles (64 rows), blocks (4 and 16
waves) and slices (64 / k rounded up to a power of two)."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


SHAPES = [
    (1, 1, 1), (63, 3, 2), (64, 4, 3), (65, 2, 9), (257, 3, 57), (1000, 8, 33), (5001, 5, 17), (70000, 16, 21),
    (65537, 11, 5), (150000, 3, 64), (150001, 7, 64), (600001, 4, 8), (530000, 16, 20),
]


@pytest.mark.parametrize("n,d,k,tie", [(*s, False) for s in SHAPES] + [(*s, True) for s in SHAPES if s[2] > 4])
def test_low_step_against_fp64(n, d, k, tie):
    from skmetal_amd import _bridge

    rng = np.random.default_rng(n + d + k)
    cen = rng.uniform(-10.0, 10.0, (k, d))
    X = (cen[rng.integers(0, k, n)] + rng.standard_normal((n, d))).astype(np.float32)
    C = np.ascontiguousarray(cen, dtype=np.float32)
    X[:k] = C  # every centre has a row of its own
    if tie:
        C[k - 1] = C[1]  # the lower index wins, the other cluster stays empty
    with _bridge.LloydHandle(n, d, k) as h:
        h.load(X, center=False)
        h.set_centers(C)
        h.iterate(1)
        lab, new = h.labels(), h.centers()
        assert h.info()["fused"] and not h.info()["split"]
    D = ((C.astype(np.float64) ** 2).sum(1)[None, :] - 2.0 * X.astype(np.float64) @ C.astype(np.float64).T)
    best = D.min(1)
    # fp32 dot products of d terms and one subtraction
    slack = (d + 4) * 2.0 ** -23 * (np.abs(X).astype(np.float64) @ np.abs(C).astype(np.float64).T).max(1) * 2.0 + \
        2.0 ** -23 * (C.astype(np.float64) ** 2).sum(1).max()
    assert np.all(D[np.arange(n), lab] <= best + slack)
    cnt = np.bincount(lab, minlength=k)
    if tie:
        assert cnt[k - 1] == 0
        return  # (an empty cluster takes a row out of another one's sums)
    assert np.all(cnt > 0)
    S = np.stack([np.bincount(lab, weights=X[:, c].astype(np.float64), minlength=k) for c in range(d)], 1)
    A = np.stack([np.bincount(lab, weights=np.abs(X[:, c]).astype(np.float64), minlength=k) for c in range(d)], 1)
    want = S / cnt[:, None]
    # an fp32 chain per wave (at most cnt rows of a cluster) and the fp32 result
    tol = (np.minimum(cnt, 4096)[:, None] * 2.0 ** -24 * A / cnt[:, None]) + 2.0 ** -23 * np.abs(want)
    assert np.all(np.abs(new - want) <= tol)
