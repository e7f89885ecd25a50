"""Banded rows and counts for bands of 65 to 512 diagonals (2 to 8 diagonals
per lane of the trace kernel) and one past them, whose pairs stay on the
int32 traceback: every AlignConfig kind and local, ties, widths at the
edges of a lane's share, bands that clip the matrix.  Scores, counts, rows
and window begins must equal the oracle's."""
import numpy as np
import pytest

import pyoracle as po
import seqan_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("band", [(-32, 32), (-60, 67), (-64, 64), (-90, 101), (-130, 140), (-200, 183), (-250, 261),
                                  (-300, 260)])
def test_wide_bands_match_oracle(ctx, band):
    lo, up = band
    rng = np.random.default_rng(500 + up)
    for ma, mi, ge, go in ((2, -3, -1, -5), (1, -1, -1, -1), (3, -2, -3, -2)):
        score = sa.simple_score(ma, mi, ge, go)
        sc = po.Scoring(score.table, go, ge)
        hs, vs = [], []
        while len(hs) < 24:
            n = int(rng.integers(2, 700))
            h = rng.integers(0, 4, n).astype(np.uint8)
            v = np.delete(h, np.nonzero(rng.random(n) < 0.02)[0])
            at, k = int(rng.integers(0, len(v) + 1)), int(rng.integers(0, 25))
            v = np.concatenate([v[:at], rng.integers(0, 4, k).astype(np.uint8), v[at:]])
            m = len(v)
            f = rng.random(m) < 0.1
            v[f] = rng.integers(0, 4, int(f.sum()))
            if m == 0 or not (lo < min(0, n - m) and max(0, n - m) < up):
                continue
            hs.append(h)
            vs.append(v.astype(np.uint8))
        Hs, Vs = sa.SeqSet.from_list(hs), sa.SeqSet.from_list(vs)
        for mode in (0, 9, 15, 4, sa.LOCAL):
            print("wide banded rows", band, (ma, mi, ge, go), "mode", mode, flush=True)
            out = ctx.align_rows_banded(Hs, Vs, score, lo, up, mode=mode)
            want = po.rows_batch(Hs.residues, Hs.offsets, Vs.residues, Vs.offsets, sc, mode, with_begins=True,
                                 band=(lo, up))
            for a, b in zip(out, want):
                assert np.array_equal(a, b), (mode, lo, up)
