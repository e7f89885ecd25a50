"""Calls of very different sizes on one context: their uploads and results
share the context's staging memory, which grows, is reused by smaller calls
and survives a call that failed in between.  Scores, counts and rows must
equal those of a fresh context."""
import numpy as np
import pytest

import seqan_amd as sa

pytestmark = pytest.mark.gpu
SIMPLE = sa.simple_score(2, -3, -1, -5)


def _calls(ctx, H, V):
    # (Plain form: its kernels start while the call still prepares.)
    return [ctx.align_score(H, V, SIMPLE, 9), ctx.align_score(H, V, SIMPLE, 9, flags=sa.PLAIN_PER_PAIR)
            if len(H) < 200 else None, *ctx.align_rows(H, V, SIMPLE, 0), *ctx.align_counts(H, V, SIMPLE, 15),
            ctx.align_score_banded(H, V, SIMPLE, -40, 40), ctx.align_score(H, V, SIMPLE, sa.LOCAL)]


def test_sizes_in_turn(ctx):
    other = sa.Context(0)
    try:
        for count in (3, 70000, 40, 300000, 40, 3, 5000):
            print("pairs", count, flush=True)
            H, V = sa.workload(sa.WL_DNA150, 0x5EED0001, 17 * count, min(count, 2000))
            if count > 2000:   # repeat the pairs: lists and results past 2 MB
                k = -(-count // 2000)
                H = sa.SeqSet(np.tile(H.residues, k), np.concatenate([[0], np.cumsum(np.tile(H.lengths(), k))]))
                V = sa.SeqSet(np.tile(V.residues, k), np.concatenate([[0], np.cumsum(np.tile(V.lengths(), k))]))
            got = _calls(ctx, H, V)
            with pytest.raises(sa.SqmiError):
                ctx.align_score_banded(H, V, SIMPLE, 5, 8)
            fresh = sa.Context(0)
            try:
                want = _calls(fresh, H, V)
            finally:
                fresh.close()
            for g, w in zip(got, want):
                assert (g is None and w is None) or np.array_equal(g, w)
            if count > 2000:   # every copy of a pair has the first one's score
                assert np.array_equal(got[0].reshape(-1, 2000), np.tile(got[0][:2000], (len(got[0]) // 2000, 1)))
            other.align_score(H, V, SIMPLE, 0)
    finally:
        other.close()
