"""The packed long-pair kernels where they change: each number of rows per
lane, sides on the edges of strips (64 rows per row of a lane) and of
checkpoints (128 steps), couples of unequal shapes and of one pair, scores
that grow enough to raise a strip's base many times, gaps longer than a
wave's 64 moves, gap costs whose extension exceeds the opening, chunks of
couples.  Scores, counts and rows must equal the oracle's."""
import numpy as np
import pytest

import pyoracle as po
import seqan_amd as sa

pytestmark = pytest.mark.gpu


def _pair(rng, n, m=None):
    h = rng.integers(0, 4, n).astype(np.uint8)
    if m is not None:
        return h, rng.integers(0, 4, m).astype(np.uint8)
    v = np.where(rng.random(n) < 0.06, rng.integers(0, 4, n), h).astype(np.uint8)
    for _ in range(max(1, n // 400)):
        a, k = int(rng.integers(0, len(v))), int(rng.integers(1, 150))
        v = np.concatenate([v[:a], v[a + k:]]) if rng.random() < 0.5 and len(v) > k + 300 else np.concatenate(
            [v[:a], rng.integers(0, 4, k).astype(np.uint8), v[a:]])
    return h, v


def _check(ctx, pairs, score, packed=True):
    H, V = sa.SeqSet.from_list([p[0] for p in pairs]), sa.SeqSet.from_list([p[1] for p in pairs])
    sc = po.Scoring(score.table, score.gap_open, score.gap_extend)
    want = po.rows_batch(H.residues, H.offsets, V.residues, V.offsets, sc, 0)
    s = ctx.align_score(H, V, score, 0)
    assert ctx.stats()["pairs_long_packed"] == (len(pairs) if packed else 0)
    assert np.array_equal(s, want[0])
    for name, g, w in zip(("scores", "counts", "op_off", "ops"), ctx.align_rows(H, V, score, 0), want):
        assert np.array_equal(g, w), name


@pytest.fixture(params=["4", "8", "16"])
def rows(request, monkeypatch):
    monkeypatch.setenv("SQMI_LONG_MIN_SIDE", "128")
    monkeypatch.setenv("SQMI_LONG_ALL", "1")
    monkeypatch.setenv("SQMI_LONG_ROWS", request.param)
    print("rows", request.param, flush=True)
    return int(request.param)


SCHEMES = [(2, -3, -1, -5), (1, -1, -1, -1), (5, -4, 0, -8), (3, -2, -3, -2), (9, -9, -4, -20)]


@pytest.mark.parametrize("scheme", SCHEMES)
def test_strip_and_checkpoint_edges(ctx, rows, scheme):
    rng = np.random.default_rng(31)
    strip = 64 * rows
    sides = [(128, 128), (191, strip - 1), (192, strip), (193, strip + 1), (255, 2 * strip - 1), (256, 2 * strip),
             (257, 2 * strip + 1), (1000, 150), (130, 1200)]
    pairs = [_pair(rng, n, m) for n, m in sides if m >= 128] + [_pair(rng, n) for n in (300, 1500, 3500, 640)]
    _check(ctx, pairs, sa.simple_score(*scheme))


def test_windows_and_chunks(ctx, rows, monkeypatch):
    # Walks through several windows, in chunks of one or two couples.
    monkeypatch.setenv("SQMI_TRACE_BUDGET_MB", "12")
    rng = np.random.default_rng(32)
    pairs = [_pair(rng, n) for n in (7000, 5200, 4000, 2600, 900)] + [_pair(rng, 6000, 700), _pair(rng, 700, 6000)]
    _check(ctx, pairs, sa.simple_score(2, -3, -1, -5))
