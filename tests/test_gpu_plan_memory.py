"""Host memory a context keeps between calls: after a call of 12 million pairs
no more than the bound on its plan's arrays (128 MB)."""
import numpy as np
import pytest

import seqan_amd as sa

pytestmark = pytest.mark.gpu
SIMPLE = sa.simple_score(2, -3, -1, -5)


def _resident_mb():
    with open("/proc/self/status") as f:
        return next(int(line.split()[1]) for line in f if line.startswith("VmRSS")) // 1024


def test_plan_of_many_pairs_is_given_back():
    n = 12000000
    off = np.arange(n + 1, dtype=np.int64) * 6
    h = np.zeros(int(off[-1]), np.uint8)
    v = h.copy()
    v[::7] = 1
    H, V = sa.SeqSet(h, off), sa.SeqSet(v, off.copy())
    dh, dv, ds = sa.DeviceBuffer.from_array(h), sa.DeviceBuffer.from_array(v), sa.DeviceBuffer(4 * n)
    own = sa.Context(0)
    try:
        own.align_score(*sa.workload(sa.WL_DNA150, 1, 0, 1000), SIMPLE, 0)
        before = _resident_mb()
        print("pairs", n, flush=True)
        own.align_score(H, V, SIMPLE, 0, h_dev=dh.address, v_dev=dv.address, scores_dev=ds.address)
        grown = _resident_mb() - before
        got = ds.to_array(np.int32, n)
    finally:
        own.close()
        for b in (dh, dv, ds):
            b.free()
    assert np.array_equal(got[:7 * 1000], got[7 * 1000:14 * 1000])   # the mutations repeat every 7 pairs
    assert grown <= 140, grown
