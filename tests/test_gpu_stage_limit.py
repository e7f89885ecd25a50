"""Calls whose staging memory is bounded below what they would use, down to
none at all: the arrays that do not fit are copied by themselves.  Scores,
counts and rows must equal those of a context that stages everything, from
host residues small enough to be staged and larger, first calls and replays."""
import numpy as np
import pytest

import seqan_amd as sa

pytestmark = pytest.mark.gpu
SIMPLE = sa.simple_score(2, -3, -1, -5)


def _calls(ctx, H, V):
    return [ctx.align_score(H, V, SIMPLE, 9), ctx.align_score(H, V, SIMPLE, 9), ctx.align_score(H, V, SIMPLE, 9),
            *ctx.align_rows(H, V, SIMPLE, 0), *ctx.align_counts(H, V, SIMPLE, 15),
            ctx.align_score_banded(H, V, SIMPLE, -40, 40), *ctx.align_rows_banded(H, V, SIMPLE, -20, 20)]


@pytest.mark.parametrize("megabytes", ["0", "1", "3"])
def test_bounded_staging(ctx, monkeypatch, megabytes):
    own = sa.Context(0)
    try:
        for count in (3, 1500, 3000, 40000, 200000, 1500):
            print("stage", megabytes, "MB, pairs", count, flush=True)
            H, V = sa.workload(sa.WL_DNA150, 0x5EED0001, 0, min(count, 3000))
            if count > 3000:
                k = count // 2000
                H, V = (sa.SeqSet(np.tile(s.residues[:s.offsets[2000]], k),
                                  np.concatenate([[0], np.cumsum(np.tile(s.lengths()[:2000], k))])) for s in (H, V))
            monkeypatch.delenv("SQMI_STAGE_MB", raising=False)
            want = _calls(ctx, H, V)
            monkeypatch.setenv("SQMI_STAGE_MB", megabytes)
            for g, w in zip(_calls(own, H, V), want):
                assert np.array_equal(g, w)
    finally:
        own.close()
