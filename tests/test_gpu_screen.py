"""The screened E-step (k_screen + k_assign3_list) against the same E-step
without the screen: the labels, and with them centres and inertia, are the
same bit for bit whatever share of the rows the screen settles."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _blobs(n, d, k, spread, seed):
    rng = np.random.default_rng(seed)
    cen = rng.standard_normal((k, d)) * spread
    X = (cen[rng.integers(0, k, n)] + rng.standard_normal((n, d))).astype(np.float32)
    return X, np.ascontiguousarray(X[:k])


def _both(monkeypatch, X, C, steps=5, center=True):
    from skmetal_amd import _bridge

    n, d = X.shape
    k = C.shape[0]
    got = []
    for mode in "01":
        monkeypatch.setenv("SKMETAL_HIP_SCREEN", mode)
        lab = np.empty(n, np.int32)
        _bridge.kmeans_assign(X, C, lab, n, d, k)
        with _bridge.LloydHandle(n, d, k) as h:
            h.load(X, center=center)
            h.set_centers(C)
            run = h.run(steps, 0.0, strict=False)
            got.append((lab, run, h.centers(), h.labels()))
            assert h.info()["asplit"] and not h.info()["fused"]
            info = h.screen_info()
            assert info["screened"] == (mode == "1") and (info["left"] >= 0) == (mode == "1")
    (l0, r0, c0, f0), (l1, r1, c1, f1) = got
    np.testing.assert_array_equal(l0, l1)
    np.testing.assert_array_equal(f0, f1)
    np.testing.assert_array_equal(c0, c1)
    assert r0[0] == r1[0] and r0[1] == pytest.approx(r1[1], rel=1e-12)
    assert not info["off"]
    return f1, info["left"]


# every K-step count, row ends off the 32-feature and 64-row grid, one stage
# of centres, several, and more than LDS keeps (k = 2000 at 4 K steps)
@pytest.mark.parametrize("n,d,k,spread", [
    (300, 17, 300, 1.0), (777, 37, 201, 0.6), (4099, 66, 129, 0.5), (513, 128, 200, 0.2), (20011, 96, 256, 0.4),
    (33333, 125, 257, 0.1), (70001, 64, 300, 0.9), (5000, 104, 2000, 0.5), (130, 32, 130, 1.0),
    # rows of more than 128 floats: 256 x 256 units, ends off both, one
    # 64-feature stage more than whole ones
    (3000, 129, 200, 0.5), (777, 300, 257, 0.4), (20011, 768, 700, 0.3), (300, 1000, 300, 0.2), (256, 192, 256, 0.3),
    # two launches of k_screen_wide (210,944 rows and the rest)
    (212_000, 132, 20_000, 0.4),
])
def test_screen_labels_match_six_products(monkeypatch, n, d, k, spread):
    _, left = _both(monkeypatch, *_blobs(n, d, k, spread, n + d))
    assert left < 0.9 * n
    assert left > 0 or n < 512  # (a few hundred rows around as many centres: all settled)


# Rows on centres far apart are settled, rows half way between two are not.  (Of
# 20,000 x 160 with 300 centres, units of 64 centres take the third that is left,
# up to 128 units of 256, and units of 256 centres all of them.)
@pytest.mark.parametrize("n,d,k", [(20000, 48, 300), (5000, 128, 700), (20000, 160, 300), (3000, 600, 260)])
@pytest.mark.parametrize("share", [0.0, 0.3, 1.0])
def test_screen_settles_what_it_can(monkeypatch, n, d, k, share):
    rng = np.random.default_rng(n)
    C = rng.standard_normal((k, d)).astype(np.float32)
    a, b = rng.integers(0, k, n), rng.integers(0, k, n)
    X = C[a].copy()
    mid = rng.random(n) < share
    X[mid] = (0.5 * (C[a] + C[b]))[mid]
    _, left = _both(monkeypatch, X, C, steps=1)
    G = np.partition(X.astype(np.float64) @ C.T.astype(np.float64) - 0.5 * (C.astype(np.float64) ** 2).sum(1), -2, 1)
    unsettled = (G[:, -1] - G[:, -2] < 1e-4).sum()  # (a third centre may be the nearest)
    assert unsettled <= left <= unsettled + 0.1 * n


@pytest.mark.parametrize("d", [24, 150])
@pytest.mark.parametrize("kind", ["duplicates", "lattice", "large", "small", "mixed", "zeros"])
def test_screen_hard_data(monkeypatch, kind, d):
    X, C = _blobs(6000, d, 140, 0.5, 3)
    if kind == "duplicates":
        C[50], C[99] = C[3], C[0]  # ties: the lowest index wins
    elif kind == "lattice":  # exact ties all over
        rng = np.random.default_rng(4)
        X = rng.integers(0, 3, X.shape).astype(np.float32)
        C = rng.integers(0, 3, C.shape).astype(np.float32)
    elif kind == "large":
        X, C = X * np.float32(1e15), C * np.float32(1e15)
    elif kind == "small":
        X, C = X * np.float32(1e-14), C * np.float32(1e-14)
    elif kind == "mixed":
        X[:, 3] *= 1e6
        C = np.ascontiguousarray(X[:140])
    else:
        X[-50:] = 0.0
        C[7] = 0.0
    _both(monkeypatch, X, C)


@pytest.mark.parametrize("d", [40, 130])
def test_screen_non_finite_centres(monkeypatch, d):
    from skmetal_amd import _bridge

    X, C = _blobs(3000, d, 150, 0.5, 6)
    C[7], C[9] = np.nan, np.inf
    lab = [np.empty(3000, np.int32) for _ in range(2)]
    for mode in (0, 1):
        monkeypatch.setenv("SKMETAL_HIP_SCREEN", str(mode))
        _bridge.kmeans_assign(X, C, lab[mode], 3000, d, 150)
    np.testing.assert_array_equal(lab[0], lab[1])


@pytest.mark.parametrize("n,d,k", [(9000, 50, 180), (30000, 128, 140), (5000, 200, 150)])
def test_screen_relocation(monkeypatch, n, d, k):
    """Empty clusters: the farthest rows come from the screen's row minima and
    are those of the six products' minima."""
    X, C = _blobs(n, d, k, 1.0, 8)
    C[[4, 20, k - 1]] = C[0]  # ties: the lowest index takes the rows
    lab, left = _both(monkeypatch, X, C, steps=1)
    assert len(np.unique(lab)) == k and 0 < left < n // 2


# Every value rounds to bf16 by 2^-8 of itself, in the direction that moves the
# high-part product of one centre up and of the other down: the pair's screen
# gap is wrong by nearly 4 * 2^-8 ||x|| ||c||, the most there is, and of the
# wrong sign.  The bound has to leave such rows to the six products.
# So too when ||c||^2 is below fp32's range and its root bounds nothing.
@pytest.mark.parametrize("scale", [0, -80])
@pytest.mark.parametrize("d", [128, 512])
def test_screen_worst_rounding(monkeypatch, d, scale):
    up, down = 1 + 2.0**-8, 1 + 3 * 2.0**-8  # ties: to 1 and to 1 + 2^-6
    half = (d - 4) // 2
    x = np.r_[np.full(half, up), np.full(half, -down), 1, 0, 0, 0]
    c1 = np.r_[np.full(half, up), np.full(half, down), 1.2 * d * 2.0**-7, 0, 0, 0]
    c1[-4] = np.round(c1[-4] * 64) / 64
    C = np.empty((160, d), np.float32)
    C[:] = -0.9 * x * (1 - 1e-3 * np.arange(160)[:, None])
    C[70], C[7] = c1, -c1
    C *= np.float32(2.0**scale)
    X = np.repeat(x[None], 1000, 0).astype(np.float32)
    _, left = _both(monkeypatch, X, C, steps=1, center=False)
    assert left == len(X)
    from skmetal_amd import _bridge

    lab = np.empty(len(X), np.int32)  # with the screen
    _bridge.kmeans_assign(X, C, lab, len(X), d, len(C))
    assert (lab == 70).all()


# a device without memory for the screen's buffers: the six products take every
# row, in that call and in the handle's later ones, and nothing is reported
@pytest.mark.parametrize("n,d,k", [(5000, 64, 300), (5000, 200, 300)])
def test_screen_without_memory(monkeypatch, n, d, k):
    from skmetal_amd import _bridge

    X, C = _blobs(n, d, k, 0.5, 9)
    got = []
    for mode in "02":
        monkeypatch.setenv("SKMETAL_HIP_SCREEN", mode)
        lab = np.empty(n, np.int32)
        _bridge.kmeans_assign(X, C, lab, n, d, k)
        with _bridge.LloydHandle(n, d, k) as h:
            h.load(X)
            for mode in {"0": "0", "2": "21"}[mode]:
                monkeypatch.setenv("SKMETAL_HIP_SCREEN", mode)
                h.set_centers(C)
                run = h.run(4, 0.0, strict=False)
                got.append((lab, h.labels(), h.centers(), np.array(run)))
            assert _bridge.last_error() == ""
    for other in got[1:]:
        for a, b in zip(got[0], other):
            np.testing.assert_array_equal(a, b)


# Without the switch a run keeps the screen while it pays: on rows that it
# settles; not on rows far from the origin, whose norms make its bound useless;
# nor where the rows it leaves lie in one stretch of X (with rows of at most 128
# floats a few blocks' work).  Labels and centres are those of the six products
# either way.
@pytest.mark.parametrize("n,d,k", [(135_000, 128, 260), (70_000, 200, 520), (9_000, 400, 1100)])
@pytest.mark.parametrize("kind", ["settled", "far", "stretch"])
def test_screen_stays_while_it_pays(monkeypatch, n, d, k, kind):
    from skmetal_amd import _bridge

    rng = np.random.default_rng(n)
    C = rng.standard_normal((k, d)).astype(np.float32)
    a, b = rng.integers(0, k, n), rng.integers(0, k, n)
    X = C[a] + 0.02 * rng.standard_normal((n, d), dtype=np.float32)
    X[:k] = C
    if kind == "far":
        X, C = X + np.float32(100), C + np.float32(100)
    elif kind == "stretch":
        some = slice(k, k + n // 10)
        X[some] = 0.5 * (C[a[some]] + C[b[some]])
    got = []
    for mode in ("0", None):
        monkeypatch.setenv("SKMETAL_HIP_SCREEN", mode) if mode else monkeypatch.delenv("SKMETAL_HIP_SCREEN")
        with _bridge.LloydHandle(n, d, k) as h:
            h.load(X, center=False)
            h.set_centers(C)
            h.iterate(7)
            mid = h.labels(), h.centers(), h.screen_info()["off"]
            h.set_centers(C)
            run = h.run(7, 0.0, strict=False)
            got.append((mid[0], mid[1], h.labels(), h.centers(), np.array(run[:1])))
            info = h.screen_info()
            assert info["screened"] == (mode is None)
    for x, y in zip(*got):
        np.testing.assert_array_equal(x, y)
    # (9,000 rows of 1,100 centres: the units spread the work over the CUs, which
    # k_assign3 does not, and all of the rows take less than without the screen)
    lost = {"settled": False, "far": n != 9_000, "stretch": d <= 128}[kind]
    assert info["off"] == mid[2] == lost
    assert (info["left"] == n) == (kind == "far") and (info["left"] > 0) == (kind != "settled")


# An E-step by itself looks at its first rows and takes the rest with or without
# the screen: the six products' labels for rows that are settled, that are not,
# and where the first rows are of the other kind than the rest.
@pytest.mark.parametrize("n,d,k", [(262_200, 40, 300), (33_000, 300, 520)])
@pytest.mark.parametrize("first,rest", [("near", "near"), ("far", "far"), ("near", "far"), ("far", "near")])
def test_screen_in_an_e_step_by_itself(monkeypatch, n, d, k, first, rest):
    from skmetal_amd import _bridge

    rng = np.random.default_rng(n)
    C = rng.standard_normal((k, d)).astype(np.float32)
    a, b = rng.integers(0, k, n), rng.integers(0, k, n)
    X = C[a] + 0.02 * rng.standard_normal((n, d), dtype=np.float32)
    part = 65536 if d <= 128 else 8192  # (at up to 8 groups of 256 centres)
    for rows, kind in ((slice(0, part), first), (slice(part, n), rest)):
        if kind == "far":
            X[rows] = 0.5 * (C[a[rows]] + C[b[rows]])
    lab = [np.empty(n, np.int32) for _ in range(2)]
    monkeypatch.setenv("SKMETAL_HIP_SCREEN", "0")
    _bridge.kmeans_assign(X, C, lab[0], n, d, k)
    monkeypatch.delenv("SKMETAL_HIP_SCREEN")
    _bridge.kmeans_assign(X, C, lab[1], n, d, k)
    np.testing.assert_array_equal(lab[0], lab[1])
    assert len(np.unique(lab[0])) == k
