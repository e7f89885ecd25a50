"""A call that fails on the host between its uploads and its kernels (the
device has no room for the alignment rows it is asked to hold): it reports
out of memory, and the calls after it on the same context, whose staging
memory its uploads still use when it returns, give what a fresh context
gives."""
import ctypes

import numpy as np
import pytest

import seqan_amd as sa

pytestmark = pytest.mark.gpu
SIMPLE = sa.simple_score(2, -3, -1, -5)


def _fail(ctx, H, V):
    # Row segments spread over 16 TiB; the call allocates them before it
    # launches or writes anything.
    n = len(H)
    seg = np.zeros(n + 1, np.int64)
    seg[1:] = np.cumsum(H.lengths() + V.lengths())
    seg[-1] += 1 << 44
    h, keep_h = sa._seqs(H)
    v, keep_v = sa._seqs(V)
    sc = SIMPLE._c()
    scores, counts = np.zeros(n, np.int32), np.zeros((n, 18), np.int32)
    ops, lens = np.zeros(int(seg[-2]) + 1, np.uint8), np.zeros(n, np.int64)
    return sa.lib().sqmi_align_rows(ctx._h, ctypes.byref(h), ctypes.byref(v), ctypes.byref(sc), 0, scores.ctypes.data,
                                    counts.ctypes.data, ops.ctypes.data, seg.ctypes.data, lens.ctypes.data, 0)


@pytest.mark.parametrize("copies", [1, 150])   # 150: offsets past 2 MB, on their way at once
def test_calls_after_a_failed_one(copies):
    H, V = sa.workload(sa.WL_DNA150, 0x5EED0001, 0, 2000)
    H2 = sa.SeqSet(np.tile(H.residues, copies), np.concatenate([[0], np.cumsum(np.tile(H.lengths(), copies))]))
    V2 = sa.SeqSet(np.tile(V.residues, copies), np.concatenate([[0], np.cumsum(np.tile(V.lengths(), copies))]))
    for call in (lambda c: [c.align_score(H, V, SIMPLE, 9)], lambda c: c.align_rows(H, V, SIMPLE, 0),
                 lambda c: [c.align_score_banded(H, V, SIMPLE, -40, 40)], lambda c: [c.align_score(H2, V2, SIMPLE, 0)]):
        own, fresh = sa.Context(0), sa.Context(0)
        try:
            print("failing call, then the next", copies, flush=True)
            assert _fail(own, H2, V2) == 6
            for _ in range(2):
                for g, w in zip(call(own), call(fresh)):
                    assert np.array_equal(g, w)
        finally:
            own.close()
            fresh.close()
