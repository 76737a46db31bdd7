"""Long chains of hooks among parents that lie in LDS (kmst_union.hip): one
workgroup's solve, and dense ids.  A chain whose root is its highest id takes
about as long as one whose root is its lowest."""
import time

import numpy as np
import pytest

import kamsta_amd as k
import oracle

pytestmark = pytest.mark.gpu


def dev(torch, x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.uint32).view(np.int32)).cuda()


def band(n, width, down, closed):
    """Every vertex and the `width` after it, weights in order; closed: a ring."""
    i = np.arange(n)
    u = np.concatenate([i[:-j] for j in range(1, width + 1)] + [[0] * closed])
    v = np.concatenate([i[j:] for j in range(1, width + 1)] + [[n - 1] * closed])
    w = 2 * n - u if down else u + 1
    s, d, w = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
    o = np.lexsort((w, d, s))
    return [x[o].astype(np.uint32) for x in (s, d, w)]


def solve(torch, ctx, rec, n):
    s, d, w = rec
    exp, exp_w = oracle.kruskal(k.to_wedges(s, d, w))
    arrs = [dev(torch, x) for x in rec]
    took = []
    for algo in [k.BORUVKA, k.FILTER_BORUVKA] * 5:
        out = torch.zeros((3, n), dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        t = time.perf_counter()
        cnt, tw = ctx.solve_device(*arrs, len(s), n, *out, n, algorithm=algo)
        took.append(time.perf_counter() - t)
        got = out.cpu().numpy().view(np.uint32)
        assert (cnt, tw) == (len(exp), exp_w)
        for row, f in zip(got, ("src", "dst", "weight")):
            assert np.array_equal(row[:cnt], exp[f]), f
    return sorted(took)[5]


# one workgroup: chains of 15 to 17 hooks (a walk's steps), of its 1024 threads and
# one more, of its most vertices; dense ids from the start: the most
@pytest.mark.parametrize("n,width,closed", [
    (16, 1, 1), (17, 1, 1), (18, 1, 1), (256, 1, 1), (257, 2, 0), (1024, 2, 0), (1025, 2, 0),
    (4096, 1, 1), (8191, 1, 1), (8192, 1, 1), (4095, 8, 0), (4096, 8, 0)])
def test_either_direction(gpu, ctx, n, width, closed):
    up, down = (solve(gpu, ctx, band(n, width, x, closed), n) for x in (False, True))
    assert down < 4 * up, (up, down)
