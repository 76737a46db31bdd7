"""Wheels (kmst_union.hip): every vertex has an edge to the hub, heavier than the
rim's, so the hub takes offers from every list in every round.  The direct solve
folds them where the hub has a large share of the records, whatever its id."""
import time

import numpy as np
import pytest

import kamsta_amd as k
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,limit", [(9000, None), (1 << 17, None), (1 << 20, 1.6)])
@pytest.mark.parametrize("hub", ["lowest", "highest"])
def test_heavy_hub(gpu, ctx, n, limit, hub):
    rng = np.random.default_rng(n)
    u = np.concatenate([np.zeros(n - 1, np.int64), np.arange(1, n - 1)])
    v = np.concatenate([np.arange(1, n), np.arange(2, n)])
    w = np.concatenate([np.full(n - 1, 1000), rng.integers(2, 255, n - 2)])
    if hub == "highest":
        u, v = n - 1 - v, n - 1 - u
    s, d, w = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
    o = np.lexsort((d, s))
    s, d, w = (x[o].astype(np.uint32) for x in (s, d, w))
    exp, exp_w = oracle.kruskal(k.to_wedges(s, d, w))
    arrs = [gpu.from_numpy(x.view(np.int32)).cuda() for x in (s, d, w)]
    took = []
    for algo in [k.BORUVKA, k.FILTER_BORUVKA] * 4:
        out = gpu.zeros((3, n), dtype=gpu.int32, device="cuda")
        gpu.cuda.synchronize()
        t = time.perf_counter()
        cnt, tw = ctx.solve_device(*arrs, len(s), n, *out, n, algorithm=algo)
        took.append(time.perf_counter() - t)
        got = out.cpu().numpy().view(np.uint32)
        assert (cnt, tw) == (len(exp), exp_w)
        for row, f in zip(got, ("src", "dst", "weight")):
            assert np.array_equal(row[:cnt], exp[f]), f
    if limit and hub == "lowest":
        assert sorted(took)[4] < limit * 1e-3, took
