"""Calls that mix pairs whose row blocks run as strips of the packed kernels
with pairs on the long-pair route, whose bottom rows take more memory than
those strips: on a fresh context, where every buffer grows during the call,
the results must be those of the two kinds in calls of their own."""
import numpy as np
import pytest

import seqan_amd as sa

pytestmark = pytest.mark.gpu
SIMPLE = sa.simple_score(2, -3, -1, -5)


def _pairs(rng, lengths):
    hs = [rng.integers(0, 4, int(n)).astype(np.uint8) for n in lengths]
    vs = []
    for h in hs:
        v = h.copy()
        f = rng.random(len(v)) < 0.1
        v[f] = rng.integers(0, 4, int(f.sum()))
        vs.append(np.delete(v, rng.integers(0, len(v), 25)))
    return hs, vs


@pytest.mark.parametrize("call", ["score", "counts"])
def test_strips_beside_long_pairs(call):
    rng = np.random.default_rng(51)
    hs, vs = _pairs(rng, [5000, 30000, 4000, 27000, 700, 5500, 31000, 4500, 29000, 5200, 3000, 4800])
    long_ = [i for i, h in enumerate(hs) if len(h) > 20000]
    short = [i for i, h in enumerate(hs) if len(h) <= 20000]

    def run(keep):
        ctx = sa.Context(0)
        try:
            A, B = (sa.SeqSet.from_list([s[i] for i in keep]) for s in (hs, vs))
            out = []
            for _ in range(3):   # the second score call captures its launches, the third replays them
                out.append((ctx.align_score(A, B, SIMPLE, 0),) if call == "score" else ctx.align_counts(A, B, SIMPLE, 0))
            print("mixed", call, len(keep), "long", ctx.stats()["pairs_long"], flush=True)
            return out
        finally:
            ctx.close()

    both, a, b = run(range(len(hs))), run(short), run(long_)
    for got, x, y in zip(both, a, b):
        for g, p, q in zip(got, x, y):
            assert np.array_equal(g[short], p) and np.array_equal(g[long_], q)
