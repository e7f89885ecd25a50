"""Score calls of many short pairs whose drifted values need all 16 bits
(mismatches dearer than two gap steps; high scores): the one-pair-per-lane
kernel's 16-bit form, alone and beside pairs that stay on lane groups, with
substitution tables and DNA bytes.  Scores must equal the int32 kernel's and,
sampled, the oracle's."""
import numpy as np
import pytest

import pyoracle as po
import seqan_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths", [(1, 31), (1, 63), (4, 100)])
@pytest.mark.parametrize("scheme", [(1, -4, -1, -2), (450, -300, -50, -300), (3, -12, -2, -2)])
def test_short_pairs_of_wide_values(ctx, scheme, lengths):
    rng = np.random.default_rng(700 + lengths[1])
    count, unit = 140000 if lengths[1] < 64 else 400000, 2000
    vl = rng.integers(lengths[0], lengths[1] + 1, unit)
    hl = np.maximum(1, vl + rng.integers(-4, 5, unit))
    hs = [rng.integers(0, 4, n).astype(np.uint8) for n in hl]
    vs = [np.resize(h, m) for h, m in zip(hs, vl)]
    for v in vs:
        f = rng.random(len(v)) < 0.15
        v[f] = rng.integers(0, 4, int(f.sum()))
    H, V = (sa.SeqSet(np.tile(np.concatenate(s), count // unit),
                      np.concatenate([[0], np.cumsum(np.tile(n, count // unit))])) for s, n in ((hs, hl), (vs, vl)))
    score = sa.simple_score(*scheme)
    sc = po.Scoring(score.table, score.gap_open, score.gap_extend)
    for mode in (0, 9, 15, 4):
        print("wide lanes", scheme, lengths, "mode", mode, flush=True)
        got = ctx.align_score(H, V, score, mode)
        assert ctx.stats()["pairs_lane"] > 0
        assert np.array_equal(got, ctx.align_score(H, V, score, mode, flags=sa.FORCE_INT32))
        want = po.score_batch(np.concatenate(hs), np.concatenate([[0], np.cumsum(hl)]), np.concatenate(vs),
                              np.concatenate([[0], np.cumsum(vl)]), sc, mode)
        assert np.array_equal(got[:unit], want)
