"""The packed banded kernel (band16.hpp) where it changes: every AlignConfig
and local alignment, each number of rows per block with rings in LDS and in
memory, narrow and wide values, bands that clip the matrix or lie off its
corners, lengths around a block's rows, couples and items of unequal |H|.
Scores must equal the oracle's and the int32 kernels'."""
import numpy as np
import pytest

import pyoracle as po
import seqan_amd as sa

pytestmark = pytest.mark.gpu

MODES = list(range(16)) + [sa.LOCAL]


def _valid(n, m, lo, up, local):
    if local:
        return n >= 2 and lo <= n - 2 and up >= -(m - 2) and min(up, n) - max(lo, -m) >= 1
    return n >= 2 and lo < min(0, n - m) and up > max(0, n - m)


def _pairs(rng, count, lo, up, alpha, top, local):
    hs, vs = [], []
    while len(hs) < count:
        m = int(rng.integers(1, top)) if rng.random() < 0.6 else 47
        n = max(2, m + int(rng.integers(max(lo, -30) + 1, max(min(up, 30), max(lo, -30) + 2))))
        if not _valid(n, m, lo, up, local):
            continue
        base = rng.integers(0, alpha, n + m).astype(np.uint8)
        h, v = base[:n].copy(), base[:m].copy()
        if rng.random() < 0.3:
            v = np.roll(v, int(rng.integers(0, 6)))
        f = rng.random(m) < (0.1 if rng.random() < 0.8 else 0.9)
        v[f] = rng.integers(0, alpha, int(f.sum()))
        hs.append(h)
        vs.append(v)
    return hs, vs


def _check(ctx, hs, vs, score, mode, lo, up):
    H, V = sa.SeqSet.from_list(hs), sa.SeqSet.from_list(vs)
    print("band", lo, up, "mode", mode, len(hs), flush=True)
    got = ctx.align_score_banded(H, V, score, lo, up, mode=mode)
    assert np.array_equal(got, ctx.align_score_banded(H, V, score, lo, up, mode=mode, flags=sa.FORCE_INT32))
    sc = po.Scoring(score.table, score.gap_open, score.gap_extend)
    k = np.random.default_rng(5).permutation(len(hs))[:120]
    want = np.array([po.score_banded(hs[i], vs[i], sc, mode, lo, up) for i in k], np.int32)
    assert np.array_equal(got[k], want), (mode, k[got[k] != want][:5])


@pytest.mark.parametrize("band", [(-5, 4), (-16, 16), (-30, 40), (-100, 80)])
@pytest.mark.parametrize("scheme", [(2, -3, -1, -5), (20, -30, -20, -60), (3, -2, -3, -2), (5, -4, 0, -8), "protein"])
def test_modes_and_value_ranges(ctx, monkeypatch, band, scheme):
    monkeypatch.setenv("SQMI_BAND_PACKED", "1")
    lo, up = band
    rng = np.random.default_rng(100 + up)
    alpha, score = (24, sa.blosum62(-1, -11)) if scheme == "protein" else (4, sa.simple_score(*scheme))
    hs, vs = _pairs(rng, 400, lo, up, alpha, 200, False)
    for mode in MODES:
        _check(ctx, hs, vs, score, mode, lo, up)


@pytest.mark.parametrize("band", [(5, 40), (-40, -6), (-12, 300), (-7, 9)])
def test_local_bands_off_the_corners(ctx, monkeypatch, band):
    monkeypatch.setenv("SQMI_BAND_PACKED", "1")
    lo, up = band
    rng = np.random.default_rng(200 + up)
    hs, vs = [], []
    while len(hs) < 300:
        n, m = int(rng.integers(2, 260)), int(rng.integers(1, 260))
        if not _valid(n, m, lo, up, True):
            continue
        h = rng.integers(0, 4, n).astype(np.uint8)
        v = rng.integers(0, 4, m).astype(np.uint8)
        at = max(lo, 0) + 3
        if n > at + 20 and m > 20:
            k = min(n - at, m, 90)
            v[:k] = h[at:at + k]
        hs.append(h)
        vs.append(v)
    for score in (sa.simple_score(2, -3, -1, -5), sa.simple_score(1, -1, -1, -1)):
        _check(ctx, hs, vs, score, sa.LOCAL, lo, up)


def test_mismatching_pairs_in_narrow_bands(ctx, monkeypatch):
    # The lowest values a band can force: no residue matches, long pairs.
    monkeypatch.setenv("SQMI_BAND_PACKED", "1")
    rng = np.random.default_rng(7)
    hs = [np.zeros(int(n), np.uint8) for n in rng.integers(1500, 1510, 40)]
    vs = [np.full(1505, 1, np.uint8) for _ in hs]
    for score in (sa.simple_score(2, -3, -1, -5), sa.simple_score(5, -4, -2, -10), sa.simple_score(2, -30, -1, -29)):
        for mode in (0, 9, 15, sa.LOCAL):
            _check(ctx, hs, vs, score, mode, -13, 13)


@pytest.mark.parametrize("band", [(-10, 12), (-18, 18), (-40, 60), (-70, 90), (-110, 115), (-200, 150)])
def test_shared_items(ctx, monkeypatch, band):
    # 2, 4 and 8 waves on an item's blocks, and one (the widest band): items of
    # fewer blocks than waves, of many, several items per workgroup.
    monkeypatch.setenv("SQMI_BAND_PACKED", "1")
    lo, up = band
    rng = np.random.default_rng(300 + up)
    hs, vs = _pairs(rng, 60, lo, up, 4, 60, False)
    for m in (1, 7, 8, 130, 511, 1200):
        for _ in range(20):
            v = rng.integers(0, 4, m).astype(np.uint8)
            n = max(2, m + int(rng.integers(lo // 2, up // 2)))
            if not _valid(n, m, lo, up, False):
                continue
            hs.append(np.concatenate([v, rng.integers(0, 4, n).astype(np.uint8)])[:n])
            vs.append(v)
    for mode in (0, 9, 15, sa.LOCAL):
        _check(ctx, hs, vs, sa.simple_score(2, -3, -1, -5), mode, lo, up)
