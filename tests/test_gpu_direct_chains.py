"""Rounds of the direct solve (kmst_union.hip) whose hooks form long chains --
weights in order along paths, bands and grids -- against the oracle, through
each kind of relabel: walks, walks into the dense ids (up to 2^15 vertices),
with parallel copies, and in a later weight class."""
import numpy as np
import pytest

import kamsta_amd as k
import oracle

pytestmark = pytest.mark.gpu


def dev(torch, x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.uint32).view(np.int32)).cuda()


def symmetric(u, v, w):
    s, d, w = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
    o = np.lexsort((w, d, s))
    return s[o].astype(np.uint32), d[o].astype(np.uint32), w[o].astype(np.uint32)


def band(n, order):
    i = np.arange(n)
    u, v = np.concatenate([i[:-1], i[:-2]]), np.concatenate([i[1:], i[2:]])
    return n, u, v, {"down": (1 << 30) - u, "up": u + 1, "equal": u * 0 + 7}[order]


def grid(side, order):
    i = np.arange(side * side).reshape(side, side)
    u = np.concatenate([i[:, :-1].ravel(), i[:-1].ravel()])
    v = np.concatenate([i[:, 1:].ravel(), i[1:].ravel()])
    return side * side, u, v, {"down": (1 << 30) - u, "up": u + 1, "equal": u * 0 + 7}[order]


def ladder(n):  # one chain from end to end beside edges too heavy to take
    i = np.arange(n - 2)
    return n, np.concatenate([i, i]), np.concatenate([i + 1, i + 2]), \
        np.concatenate([(1 << 30) - i, np.full(n - 2, 0xFFFFFFF0)])


def copies(n):  # every edge of a ladder twice, of one weight
    n, u, v, w = ladder(n)
    return n, np.tile(u, 2), np.tile(v, 2), np.tile(w, 2)


def cliques(count, size):  # light cliques, heavier edges in order from one to the next
    a, b = np.triu_indices(size, 1)
    at = size * np.arange(count)[:, None]
    j = size * np.arange(count - 1)
    rng = np.random.default_rng(count)
    return count * size, np.concatenate([(a + at).ravel(), j]), np.concatenate([(b + at).ravel(), j + size]), \
        np.concatenate([rng.integers(1, 1000, len(a) * count), (1 << 30) - np.arange(count - 1)])


CASES = {
    "band down 8193": (band, 8193, "down"), "band down 20000": (band, 20000, "down"),
    "band down 32768": (band, 32768, "down"), "band down 32769": (band, 32769, "down"),
    "band down 300000": (band, 300000, "down"), "band up 40000": (band, 40000, "up"),
    "band equal 40000": (band, 40000, "equal"), "grid down 120": (grid, 120, "down"),
    "grid down 700": (grid, 700, "down"), "grid equal 300": (grid, 300, "equal"),
    "ladder 10000": (ladder, 10000), "ladder 40000": (ladder, 40000), "ladder 1500000": (ladder, 1500000),
    "copies 9000": (copies, 9000), "copies 50000": (copies, 50000),
    "cliques 3000": (cliques, 3000, 20), "cliques 20000": (cliques, 20000, 14),
}


@pytest.mark.parametrize("name", CASES)
def test_chains(gpu, ctx, name):
    make, *args = CASES[name]
    n, u, v, w = make(*args)
    s, d, w = symmetric(u, v, w)
    exp, exp_w = oracle.kruskal(k.to_wedges(s, d, w))
    rec = [dev(gpu, x) for x in (s, d, w)]
    gpu.cuda.synchronize()
    for algo in (k.BORUVKA, k.FILTER_BORUVKA):
        for _ in range(2):
            out = gpu.zeros((3, n), dtype=gpu.int32, device="cuda")
            gpu.cuda.synchronize()
            cnt, tw = ctx.solve_device(*rec, len(s), n, *out, n, algorithm=algo)
            got = out.cpu().numpy().view(np.uint32)
            assert (cnt, tw) == (len(exp), exp_w)
            for row, f in zip(got, ("src", "dst", "weight")):
                assert np.array_equal(row[:cnt], exp[f]), f
                assert not row[cnt:].any()
        rounds = ctx.stats()["rounds"]
        assert all(r["direct"] != r["chains"] for r in rounds)  # the direct solve's, of either kind
        if "down" in name or "ladder" in name or "copies" in name or "cliques" in name:
            assert any(r["chains"] for r in rounds)


def test_random_weights_walk(gpu, ctx):
    for n, m in ((9000, 45000), (1 << 17, 1 << 20)):
        rec = [dev(gpu, x) for x in k.gen_gnm_host(n, m, 254, 7)]
        out = gpu.zeros((3, n), dtype=gpu.int32, device="cuda")
        gpu.cuda.synchronize()
        ctx.solve_device(*rec, 2 * m, n, *out, n)
        assert all(r["direct"] and not r["chains"] for r in ctx.stats()["rounds"])
