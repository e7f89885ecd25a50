"""Banded scores under a free first row with substitution schemes whose scores
are all negative: there a gap may cost 256 and more while the diagonal's
scores still fit the packed kernel's DNA bytes, and the score that holds row
0 at 0 (the gap's cost) does not.  Every AlignConfig and local, against the
oracle and the int32 kernels, with gap costs on both sides of a byte's 255."""
import numpy as np
import pytest

import pyoracle as po
import seqan_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("band", [(-10, 10), (-30, 25), (-70, 75)])
@pytest.mark.parametrize("scheme", [(-3, -4, -1, -254), (-3, -4, -1, -255), (-2, -4, -1, -256), (-3, -4, -1, -257),
                                    (-5, -6, -1, -258), (-200, -300, -10, -444)])
def test_gap_costs_around_a_byte(ctx, monkeypatch, scheme, band):
    monkeypatch.setenv("SQMI_BAND_PACKED", "1")
    lo, up = band
    rng = np.random.default_rng(900 - scheme[3] + up)
    score = sa.simple_score(*scheme)
    sc = po.Scoring(score.table, score.gap_open, score.gap_extend)
    hs, vs = [], []
    while len(hs) < 150:
        m = int(rng.integers(1, 90))
        n = m + int(rng.integers(-8, 9))
        if n < 2 or not (lo < min(0, n - m) and max(0, n - m) < up):
            continue
        h = rng.integers(0, 4, n).astype(np.uint8)
        v = np.resize(h, m)
        f = rng.random(m) < 0.2
        v[f] = rng.integers(0, 4, int(f.sum()))
        hs.append(h)
        vs.append(v)
    H, V = sa.SeqSet.from_list(hs), sa.SeqSet.from_list(vs)
    for mode in list(range(16)) + [sa.LOCAL]:
        print("band", band, scheme, "mode", mode, flush=True)
        got = ctx.align_score_banded(H, V, score, lo, up, mode=mode)
        assert ctx.stats()["pairs_int16"] > 100   # the packed route
        want = np.array([po.score_banded(h, v, sc, mode, lo, up) for h, v in zip(hs, vs)], np.int32)
        assert np.array_equal(got, want), (mode, int((got != want).sum()))
        assert np.array_equal(got, ctx.align_score_banded(H, V, score, lo, up, mode=mode, flags=sa.FORCE_INT32))
