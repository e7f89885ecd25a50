"""Score calls whose pairs' row blocks would take more device memory as strips
than the budget holds: the items past it are swept whole, the scores stay the
same and the context's memory stays bounded."""
import ctypes

import numpy as np
import pytest

import pyoracle as po
import seqan_amd as sa

pytestmark = pytest.mark.gpu
SIMPLE = sa.simple_score(2, -3, -1, -5)


def _free():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert sa.hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def _pairs(rng, count, lo, hi):
    hs = [rng.integers(0, 4, int(n)).astype(np.uint8) for n in rng.integers(lo, hi + 1, count)]
    vs = []
    for h in hs:
        v = h.copy()
        f = rng.random(len(v)) < 0.1
        v[f] = rng.integers(0, 4, int(f.sum()))
        vs.append(np.delete(v, rng.integers(0, len(v), 30)))
    return sa.SeqSet.from_list(hs), sa.SeqSet.from_list(vs)


def test_strips_stay_within_their_budget(ctx, monkeypatch):
    # 200 couples of 24 blocks x 12,000 columns x 8 bytes: 460 MB of strips.
    rng = np.random.default_rng(31)
    H, V = _pairs(rng, 400, 11500, 12000)
    want = ctx.align_score(H, V, SIMPLE, 9)
    monkeypatch.setenv("SQMI_TRACE_BUDGET_MB", "16")
    own = sa.Context(0)
    try:
        before = _free()
        got = own.align_score(H, V, SIMPLE, 9)
        grown = before - _free()
    finally:
        own.close()
    print("device memory of the call:", grown >> 20, "MB", flush=True)
    assert np.array_equal(got, want)
    assert grown < 256 << 20, grown


@pytest.mark.parametrize("mode", [0, 9, 15, sa.LOCAL])
def test_whole_items_beside_strips(ctx, monkeypatch, mode):
    # Longest first: strips, whole items, strips again, by a budget of 1 MB.
    rng = np.random.default_rng(32 + mode)
    H, V = _pairs(rng, 60, 700, 2600)
    monkeypatch.setenv("SQMI_TRACE_BUDGET_MB", "1")
    got = ctx.align_score(H, V, SIMPLE, mode)
    want = po.score_batch(H.residues, H.offsets, V.residues, V.offsets,
                          po.Scoring(SIMPLE.table, SIMPLE.gap_open, SIMPLE.gap_extend), mode)
    assert np.array_equal(got, want)
