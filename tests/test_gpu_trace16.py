"""The packed trace kernel and the 16-lane walk where they change: row blocks
of an item on different waves, wide values, gap costs whose extension exceeds
the opening (every gap character reopens), long gaps (more than 16 equal
moves), ends on row and block edges.  Scores, counts and rows must equal the
oracle's."""
import numpy as np
import pytest

import pyoracle as po
import seqan_amd as sa

pytestmark = pytest.mark.gpu


def _gapped(rng, n, alpha):
    """H of length n and V: a copy with substitutions and a few gaps of up to 60."""
    h = rng.integers(0, alpha, n).astype(np.uint8)
    v = np.where(rng.random(n) < 0.1, rng.integers(0, alpha, n), h).astype(np.uint8)
    for _ in range(max(1, n // 250)):
        a, k = int(rng.integers(0, len(v))), int(rng.integers(1, 60))
        v = np.concatenate([v[:a], v[a + k:]]) if rng.random() < 0.5 and len(v) > k + 1 else np.concatenate(
            [v[:a], rng.integers(0, alpha, k).astype(np.uint8), v[a:]])
    return h, v


def _set(rng, lengths, alpha=4):
    pairs = [_gapped(rng, n, alpha) for n in lengths]
    return sa.SeqSet.from_list([p[0] for p in pairs]), sa.SeqSet.from_list([p[1] for p in pairs])


def _check_rows(ctx, H, V, score, mode):
    print("mode", mode, flush=True)
    sc = po.Scoring(score.table, score.gap_open, score.gap_extend)
    if mode & sa.LOCAL:
        got = ctx.align_local_rows(H, V, score)
        want = po.rows_batch(H.residues, H.offsets, V.residues, V.offsets, sc, sa.LOCAL, with_begins=True)
    else:
        got = ctx.align_rows(H, V, score, mode)
        want = po.rows_batch(H.residues, H.offsets, V.residues, V.offsets, sc, mode)
    for name, g, w in zip(("scores", "counts", "op_off", "ops", "begins"), got, want):
        assert np.array_equal(g, w), (mode, name)


SCHEMES = [(2, -3, -1, -5), (20, -30, -20, -60), (1, -1, -1, -1), (4, -2, -6, -3), (3, -40, -1, -2), (5, -4, 0, -8)]


@pytest.mark.parametrize("scheme", SCHEMES)
def test_rows_on_edges_and_ranges(ctx, scheme):
    rng = np.random.default_rng(11)
    lengths = [1, 2, 16, 17, 63, 64, 254, 255, 256, 257, 300, 510, 511, 512, 513, 700, 1100]
    H, V = _set(rng, lengths)
    score = sa.simple_score(*scheme)
    for mode in (0, 9, 15, 4, 2, sa.LOCAL):
        _check_rows(ctx, H, V, score, mode)


@pytest.mark.parametrize("min_blocks", ["0", "2"])
def test_whole_items_and_strips(ctx, monkeypatch, min_blocks):
    monkeypatch.setenv("SQMI_COOP_MIN_BLOCKS", min_blocks)
    rng = np.random.default_rng(12)
    H, V = _set(rng, [int(x) for x in rng.integers(100, 1500, 40)])
    for mode in (0, 9, 15, sa.LOCAL):
        _check_rows(ctx, H, V, sa.simple_score(2, -3, -1, -5), mode)
    P, Q = _set(rng, [900, 400, 300, 1200], 24)
    for mode in (0, 15, sa.LOCAL):
        _check_rows(ctx, P, Q, sa.blosum62(-1, -11), mode)


def test_counts_in_chunks_with_strips(ctx, monkeypatch):
    # Trace records of a chunk at most 2 MB: several chunks, each with strips.
    monkeypatch.setenv("SQMI_TRACE_BUDGET_MB", "2")
    rng = np.random.default_rng(13)
    H, V = _set(rng, [int(x) for x in rng.integers(200, 900, 60)])
    score = sa.simple_score(2, -3, -1, -5)
    for mode in (0, 9, 15, sa.LOCAL):
        _check_rows(ctx, H, V, score, mode)


def test_local_best_in_an_early_block(ctx, monkeypatch):
    # Whole items of several row blocks whose best cell lies in the first
    # ones: a later block's lower cells must not replace it.
    monkeypatch.setenv("SQMI_COOP_MIN_BLOCKS", "0")
    rng = np.random.default_rng(14)
    for alpha, score in ((4, sa.simple_score(2, -3, -1, -5)), (24, sa.blosum62(-1, -11))):
        hs, vs = [], []
        for n in (300, 600, 900, 1200):
            for at in (0, n // 3, n - 120):
                h, v = (rng.integers(0, alpha, n).astype(np.uint8) for _ in range(2))
                v[at:at + 60] = h[n // 2:n // 2 + 60]
                hs.append(h)
                vs.append(v)
        _check_rows(ctx, sa.SeqSet.from_list(hs), sa.SeqSet.from_list(vs), score, sa.LOCAL)


@pytest.mark.parametrize("budget", ["", "2"])
@pytest.mark.parametrize("lanes", ["16", "64"])
def test_lanes_per_couple(ctx, monkeypatch, lanes, budget):
    # Both forms of the trace kernel for every item, in one chunk and several;
    # lengths around a block (256 rows) and a lane's rows (4 and 16).
    monkeypatch.setenv("SQMI_TRACE_LANES", lanes)
    if budget:
        monkeypatch.setenv("SQMI_TRACE_BUDGET_MB", budget)
    rng = np.random.default_rng(15)
    lengths = [1, 3, 4, 5, 15, 16, 17, 63, 64, 65, 250, 254, 255, 256, 257, 260, 511, 512, 700, 1300]
    H, V = _set(rng, lengths)
    for scheme in ((2, -3, -1, -5), (20, -30, -20, -60), (4, -2, -6, -3)):
        for mode in (0, 9, 15, 2, 4, sa.LOCAL):
            _check_rows(ctx, H, V, sa.simple_score(*scheme), mode)
    P, Q = _set(rng, [900, 400, 300, 1200, 255, 31], 24)
    for mode in (0, 15, sa.LOCAL):
        _check_rows(ctx, P, Q, sa.blosum62(-1, -11), mode)
