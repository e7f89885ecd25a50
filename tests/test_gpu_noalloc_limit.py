"""The no-allocation call near the end of its 64 MiB scratch array: a call of
pairs in device memory needs two offsets and an order entry per pair and 16
bytes per eight pairs (16 lanes per couple), and is accepted while these fit,
protein tables included; a few pairs more are refused."""
import numpy as np
import pytest

import seqan_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("residues", ["dna", "protein"])
def test_lists_that_nearly_fill_the_scratch(ctx, residues):
    dna = residues == "dna"
    score = sa.simple_score(2, -3, -1, -5) if dna else sa.blosum62(-1, -11)
    rng = np.random.default_rng(41)
    n = 3000000      # 22 bytes a pair: 66.0e6 of 67.1e6
    unit = 5000
    m = rng.integers(5, 12, unit)
    lens = np.tile(m, n // unit)
    off = np.zeros(n + 1, np.int64)
    off[1:] = np.cumsum(lens)
    h = np.tile(rng.integers(0, 4 if dna else 20, int(m.sum())).astype(np.uint8), n // unit)
    v = h.copy()
    f = rng.random(len(v)) < 0.2
    v[f] = 1
    H, V = sa.SeqSet(h, off), sa.SeqSet(v, off.copy())
    dh, dv, ds = sa.DeviceBuffer.from_array(h), sa.DeviceBuffer.from_array(v), sa.DeviceBuffer(4 * n)
    flags = sa.force_shape(16, 16)
    try:
        print("noalloc", residues, n, flush=True)
        ctx.align_score_noalloc(H, V, score, 0, flags=flags, h_dev=dh.address, v_dev=dv.address, scores_dev=ds.address)
        got = ds.to_array(np.int32, n)
        ctx.align_score(H, V, score, 0, flags=flags, h_dev=dh.address, v_dev=dv.address, scores_dev=ds.address)
        assert np.array_equal(got, ds.to_array(np.int32, n))
    finally:
        for b in (dh, dv, ds):
            b.free()
