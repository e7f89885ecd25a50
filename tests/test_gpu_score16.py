"""The packed score kernel where its value range, its block shapes and its
split over waves change: values at and past the three-operand maximum's range
(wide values), scores below the gap costs, costly gap extensions, row counts
at the edges of row units and blocks, and long pairs whose row blocks go to
different waves.  All scores are integers and must equal the oracle's."""
import numpy as np
import pytest

import pyoracle as po
import seqan_amd as sa

pytestmark = pytest.mark.gpu

EDGES = (1, 2, 15, 16, 17, 63, 64, 65, 127, 128, 191, 192, 255, 256, 257, 383, 384, 511, 512, 513)


def _set(rng, lengths, alpha, related=True):
    hs, vs = [], []
    for n, m in lengths:
        h = rng.integers(0, alpha, n).astype(np.uint8)
        v = rng.integers(0, alpha, m).astype(np.uint8)
        if related:
            k = min(n, m)
            v[:k] = np.where(rng.random(k) < 0.85, h[:k], v[:k])
        hs.append(h)
        vs.append(v)
    return sa.SeqSet.from_list(hs), sa.SeqSet.from_list(vs)


def _check(ctx, H, V, score, mode, **kw):
    print("mode", mode, kw, flush=True)
    got = ctx.align_score(H, V, score, mode, **kw)
    want = po.score_batch(H.residues, H.offsets, V.residues, V.offsets,
                          po.Scoring(score.table, score.gap_open, score.gap_extend), mode)
    assert np.array_equal(got, want), (mode, np.nonzero(got != want)[0][:8])


# (match, mismatch, extend, open): the usual scheme; wide values from 320 bp
# on; t of a mismatch below 0 (table path); linear gaps; an extension costlier
# than an opening; free extension; costly extension (local drift).
SCHEMES = [(2, -3, -1, -5), (40, -30, -20, -60), (3, -40, -1, -2), (1, -1, -1, -1), (4, -2, -6, -3), (5, -4, 0, -8),
           (100, -90, -90, -95)]


@pytest.mark.parametrize("scheme", SCHEMES)
def test_value_ranges_and_row_edges(ctx, scheme):
    rng = np.random.default_rng(abs(hash(scheme)) % 1000)
    edges = [(int(rng.integers(1, 280)), m) for m in EDGES] + [(n, int(rng.integers(1, 280))) for n in EDGES]
    H, V = _set(rng, edges, 4)
    score = sa.simple_score(*scheme)
    for mode in (0, 9, 15, 4, 2, sa.LOCAL):
        _check(ctx, H, V, score, mode)
        _check(ctx, H, V, score, mode, flags=sa.force_shape(16, 16))


@pytest.mark.parametrize("gaps", [(-1, -11), (-1, -2), (-30, -40)])
def test_table_scores(ctx, gaps):
    rng = np.random.default_rng(7)
    edges = [(int(rng.integers(1, 400)), m) for m in EDGES]
    H, V = _set(rng, edges, 24)
    score = sa.blosum62(*gaps)
    for mode in (0, 9, 15, sa.LOCAL):
        _check(ctx, H, V, score, mode)
        _check(ctx, H, V, score, mode, flags=sa.force_shape(16, 16))


@pytest.mark.parametrize("count", [1, 2, 5])
def test_long_pairs_in_strips(ctx, count):
    # A few long pairs: every row block goes to its own wave.
    rng = np.random.default_rng(count)
    lengths = [(int(rng.integers(900, 3200)), int(rng.integers(900, 3200))) for _ in range(count)] + [(40, 30)]
    H, V = _set(rng, lengths, 4)
    for scheme in ((2, -3, -1, -5), (6, -4, -3, -8)):
        for mode in (0, 9, 15, sa.LOCAL):
            _check(ctx, H, V, sa.simple_score(*scheme), mode)
    P, Q = _set(rng, [(700, 1900), (1500, 1200)], 24)
    _check(ctx, P, Q, sa.blosum62(-1, -11), sa.LOCAL)
    _check(ctx, P, Q, sa.blosum62(-1, -11), 0)


def test_strips_of_many_pairs(ctx, monkeypatch):
    # More strips than the chip holds waves, 16 and 64 lanes, and one pair
    # much longer than the rest.
    rng = np.random.default_rng(3)
    lengths = [(int(rng.integers(300, 700)), int(rng.integers(300, 700))) for _ in range(6000)] + [(2900, 3000)]
    H, V = _set(rng, lengths, 4)
    score = sa.simple_score(2, -3, -1, -5)
    _check(ctx, H, V, score, 9)
    monkeypatch.setenv("SQMI_COOP_MIN_BLOCKS", "2")
    _check(ctx, H, V, score, 9, flags=sa.force_shape(64, 4))
    _check(ctx, H, V, score, sa.LOCAL, flags=sa.force_shape(16, 8))
