"""Which score calls the planner gives to the one-pair-per-lane kernels."""
import numpy as np
import pytest

import seqan_amd as sa


def _short_pairs(count):
    lens = np.tile(np.arange(30, 41), count // 11 + 1)[:count]
    off = np.zeros(count + 1, np.int64)
    off[1:] = np.cumsum(lens)
    res = np.zeros(int(off[-1]), np.uint8)
    return sa.SeqSet(res, off), sa.SeqSet(res.copy(), off.copy())


@pytest.mark.parametrize("mode", [0, 9, 15, sa.LOCAL])
@pytest.mark.parametrize("scheme", [(2, -3, -1, -5), (1, -4, -1, -2), (2, -3, -5, -2)])
def test_many_short_pairs_take_lanes_under_every_scheme(scheme, mode):
    # 1/-4/-1/-2: a mismatch costs more than two gap steps, so the drifted
    # scores are negative and take the lane kernel's 16-bit form.
    H, V = _short_pairs(524288)
    st = sa.plan_stats(H, V, sa.simple_score(*scheme), mode=mode)
    assert st["pairs_lane"] == st["pairs_int16"] == 524288


@pytest.mark.parametrize("mode", [0, sa.LOCAL])
def test_a_few_thousand_short_pairs_stay_on_16_lanes(mode):
    # Eight pairs per item; on 64 lanes, two per item, claiming four times the
    # items takes longer than their shorter sweeps save.
    rng = np.random.default_rng(4)
    lens = rng.integers(20, 61, 4096)
    off = np.zeros(4097, np.int64)
    off[1:] = np.cumsum(lens)
    res = np.zeros(int(off[-1]), np.uint8)
    st = sa.plan_stats(sa.SeqSet(res, off), sa.SeqSet(res.copy(), off.copy()), sa.simple_score(2, -3, -1, -5), mode=mode)
    assert st["work_items"] <= 600
