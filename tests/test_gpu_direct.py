"""The direct solve (kmst_union.hip), one launch for a whole graph: sizes at the
edges of its units (256 records), waves, workgroups and chunks, arrays at every
word alignment, graphs with ties, parallel records, long chains and one
component that most edges touch, against the oracle; malformed inputs keep the
round loop's status."""
import dataclasses

import numpy as np
import pytest

import kamsta_amd as k
import oracle

pytestmark = pytest.mark.gpu


def dev(torch, x, pad=0):
    """The array on the device, `pad` words past the start of its allocation."""
    whole = torch.empty(len(x) + pad, dtype=torch.int32, device="cuda")
    whole[pad:] = torch.from_numpy(np.ascontiguousarray(x, dtype=np.uint32).view(np.int32))
    return whole[pad:]


def symmetric(u, v, w):
    s, d, w = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
    o = np.lexsort((w, d, s))
    return s[o].astype(np.uint32), d[o].astype(np.uint32), w[o].astype(np.uint32)


def check(torch, ctx, s, d, w, n, pads=((0, 0, 0),), direct=True, algos=(k.BORUVKA, k.FILTER_BORUVKA)):
    rec = k.to_wedges(s, d, w)
    exp, exp_w = oracle.kruskal(rec) if len(s) < 1 << 23 else oracle.boruvka(rec, 1, 8)
    for pad in pads:
        rec = [dev(torch, x, p) for x, p in zip((s, d, w), pad)]
        for algo in algos:
            out = torch.zeros((3, n), dtype=torch.int32, device="cuda")
            cnt, tw = ctx.solve_device(*rec, len(s), n, *out, n, algorithm=algo)
            got = out.cpu().numpy().view(np.uint32)
            assert (cnt, tw) == (len(exp), exp_w), (n, len(s), pad, algo)
            for row, f in zip(got, ("src", "dst", "weight")):
                assert np.array_equal(row[:cnt], exp[f]), (n, len(s), pad, algo, f)
                assert not row[cnt:].any()
            if direct is not None:
                assert any(r.get("direct") for r in ctx.stats()["rounds"]) == direct


# undirected edges of a GNM graph on n vertices: half a unit, one unit, one
# workgroup's first and last units, two workgroups, a chunk's first record
@pytest.mark.parametrize("n,edges", [
    # one workgroup in registers and LDS up to 2^14 records and 2^13 vertices
    (3, 3), (40, 511), (40, 512), (40, 513), (200, 8191), (200, 8192), (200, 8193),
    (8191, 8191), (8192, 8192), (8193, 8193),
    (16, 100), (17, 127), (17, 128), (17, 129), (64, 1000), (256, 4095), (256, 4096), (256, 4097),
    (300, 16 * 256), (1000, 8193), (4097, 65537), (65535, 1 << 17), (65536, (1 << 17) + 1),
    # dense ids from the start up to 4096 vertices
    (4095, 30000), (4096, 30000), (4097, 30000), (5000, 300000), (9000, 36001),
    (100003, (1 << 21) - 1), (100003, 1 << 21), (100003, (1 << 21) + 129)])
def test_sizes_and_alignment(gpu, ctx, n, edges):
    s, d, w = k.gen_gnm_host(n, edges, 254, edges)
    pads = ((0, 0, 0), (1, 2, 3)) if edges < 1 << 20 else ((3, 0, 1),)
    check(gpu, ctx, s, d, w, n, pads)


def shape(name):
    rng = np.random.default_rng(11)
    if name == "pair":  # every record of a two-vertex multigraph is parallel
        return 2, np.zeros(40, int), np.ones(40, int), rng.integers(1, 4, 40)
    if name == "triangle":
        return 3, np.array([0, 0, 1]), np.array([1, 2, 2]), np.array([7, 7, 7])
    if name == "ring":  # exactly 2 n records; increasing weights hook one long chain
        i = np.arange(50000)
        return 50000, np.minimum(i, (i + 1) % 50000), np.maximum(i, (i + 1) % 50000), i + 1
    if name == "ladder":  # a chain beside edges too heavy to take
        i = np.arange(30000)
        return 30002, np.concatenate([i, i]), np.concatenate([i + 1, i + 2]), \
            np.concatenate([30000 - i, np.full(30000, 0xFFFFFFF0)])
    if name == "parallel":
        u, v = rng.integers(0, 3000, 40000), rng.integers(0, 3000, 40000)
        u, v = np.minimum(u, v)[u != v], np.maximum(u, v)[u != v]
        return 3000, np.concatenate([u, u]), np.concatenate([v, v]), rng.integers(1, 5, 2 * len(u))
    if name == "equal":  # all weights alike: every edge is light
        u, v = np.triu_indices(300, 1)
        return 300, u, v, np.full(len(u), 9)
    if name == "extremes":  # weights 0 and 2^32 - 1, isolated vertices at both ends
        u, v = np.triu_indices(200, 1)
        return 900, u + 300, v + 300, np.where(rng.integers(0, 2, len(u)) > 0, 0xFFFFFFFF, 0)
    if name == "islands":  # 500 cliques: no component is a giant
        u, v = np.triu_indices(20, 1)
        at = 20 * np.arange(500)[:, None]
        return 10000, (u + at).ravel(), (v + at).ravel(), rng.integers(1, 1 << 31, 500 * len(u))
    if name == "hubs":  # four vertices of degree n
        n = 30000
        u = np.repeat(np.arange(4), n - 4)
        v = np.tile(np.arange(4, n), 4)
        return n, u, v, rng.integers(1, 255, len(u))
    if name == "gap":  # 40000 ids without records inside a row of 2048 positions
        u, v = np.triu_indices(300, 1)
        far = lambda x: np.where(x < 150, x, x + 40000)
        return 40150 + 150, far(u), far(v), rng.integers(1, 255, len(u))
    if name in ("outer hub", "outer rows"):  # a dense block, and beside it rows of 5000 / 40 records
        u, v = rng.integers(0, 9000, 200000), rng.integers(0, 9000, 200000)
        u, v = np.unique(np.stack([np.minimum(u, v), np.maximum(u, v)])[:, u != v], axis=1)
        wheels = 1 if name == "outer hub" else 100
        rim = np.arange(5000 // wheels if wheels == 1 else 40)
        size = len(rim) + 1
        at = 9000 + size * np.arange(wheels)[:, None]
        u = np.concatenate([u, (at + 0 * rim).ravel(), (at + 1 + rim[:-1]).ravel()])
        v = np.concatenate([v, (at + 1 + rim).ravel(), (at + 2 + rim[:-1]).ravel()])
        return 9000 + wheels * size, u, v, rng.integers(1, 255, len(u))
    raise KeyError(name)


@pytest.mark.parametrize("name", ["pair", "triangle", "ring", "ladder", "parallel", "equal", "extremes",
                                  "islands", "hubs", "gap", "outer hub", "outer rows"])
def test_shapes(gpu, ctx, name):
    n, u, v, w = shape(name)
    # one chain of 30000 hooks: the direct solve gives up, the round loop solves
    check(gpu, ctx, *symmetric(u, v, w), n, direct={"ladder": False, "ring": None}.get(name, True))


def test_rule(gpu, ctx):
    """Fewer than two records per vertex: the round loop.  From 2^18 and from 2^21
    vertices on one and two more light classes."""
    i = np.arange(999)
    check(gpu, ctx, *symmetric(i, i + 1, i % 7 + 1), 1000, direct=False)
    for n, phases in ((1 << 18) - 1, 2), (1 << 18, 3), ((1 << 21) - 1, 3), (1 << 21, 4):
        s, d, w = k.gen_gnm_host(n, 4 * n, 254, n)
        check(gpu, ctx, s, d, w, n, algos=(k.BORUVKA,))
        assert len(ctx.stats()["filter"]) == phases, n


@pytest.mark.parametrize("edges", [500, 40000])
@pytest.mark.parametrize("fault", ["order", "id", "loop", "odd", "twin", "weight", "room"])
def test_refused_as_by_the_round_loop(gpu, ctx, edges, fault):
    n = 200 if edges == 500 else 4000
    s, d, w = (x.copy() for x in k.gen_gnm_host(n, edges, 254, 5))
    m, cap, at = len(s), n, len(s) // 2 + 3
    if fault == "order":
        s[at], s[-1] = s[-1], s[at]
    elif fault == "id":
        s[-1] = n
    elif fault == "loop":
        d[at] = s[at]
    elif fault == "odd":
        s, d, w, m = s[:-1], d[:-1], w[:-1], m - 1
    elif fault == "twin":
        d[-1] = d[-1] - 1 if d[-1] - 1 != d[-2] else d[-1] + 1
    elif fault == "weight":
        w[at] += 1
    elif fault == "room":
        cap = 3
    status = []
    entry = ctx.get_tuning()
    for limit in (entry.persistent_max, 0):  # 0: the round loop
        try:
            ctx.set_tuning(dataclasses.replace(entry, persistent_max=limit))
            out = gpu.zeros((3, n), dtype=gpu.int32, device="cuda")
            with pytest.raises(k.KmstError) as e:
                ctx.solve_device(*(dev(gpu, x) for x in (s, d, w)), m, n, *out, cap)
            status.append(e.value.status)
            assert not out[:, cap:].any()
        finally:
            ctx.set_tuning(entry)
    assert status[0] == status[1], (fault, status)
    # the context goes on
    s, d, w = k.gen_gnm_host(n, edges, 254, 6)
    check(gpu, ctx, s, d, w, n)


@pytest.mark.parametrize("copy", ["0", "1"])
def test_read_back(gpu, copy, monkeypatch):
    """Counters published to mapped host memory, or copied."""
    monkeypatch.setenv("KMST_READBACK_COPY", copy)
    s, d, w = k.gen_gnm_host(5000, 40000, 254, 3)
    own = k.Context()
    check(gpu, own, s, d, w, 5000)
    own.close()
