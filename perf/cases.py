"""The workloads whose speed this repository looks after.

Each case is one call (or, for the server, one burst of requests) as a program
that uses the library makes it: a minimum spanning forest of one graph through
the device, the host or the no-allocation entry point, or of many graphs
through the batched server.  Graphs come from the library's deterministic
generators (GNM, RGG2D, RHG); sizes run from the smallest serving request
(2^8 vertices) to the headline graph (2^24 vertices, 2^28 edges).

A case holds plain values: what it calls (`via`), the algorithm, the graph
(`graph`, `n`, `m` undirected edges or `degree` directed records per vertex),
the largest weight (31-bit weights leave no room for the vertex ids in one
64-bit key, which takes the library's other key format), and the options.
"""
import math

import numpy as np
import torch

import kamsta_amd as k

W8 = 254             # the reference's experiments: weights U[1, 254]
W31 = (1 << 31) - 1
EXACT_RECORDS = 1 << 21   # inputs of at most this many records have an exact()


def listed():
    return [
        # the smallest request that the serving workload has: latency alone
        {"name": "gnm_2e8_plain", "via": "device", "algorithm": "boruvka", "graph": "gnm",
         "n": 300, "m": 2205, "max_weight": W8, "threshold": 4},
        # the reference's CPU-sized configuration
        {"name": "gnm_2e14_plain", "via": "device", "algorithm": "boruvka", "graph": "gnm",
         "n": 1 << 14, "m": 1 << 18, "max_weight": W8, "threshold": 4},
        # a caller that may not allocate, near the limits of that entry point
        {"name": "gnm_40k_noalloc", "via": "noalloc", "algorithm": "filter_boruvka",
         "graph": "gnm", "n": 40009, "m": 400077, "max_weight": W8, "threshold": 4},
        # one core's share of the reference's weak scaling runs
        {"name": "gnm_2e17_filter", "via": "device", "algorithm": "filter_boruvka",
         "graph": "gnm", "n": 1 << 17, "m": 1 << 20, "max_weight": W8, "threshold": 4},
        # an ordinary geometric graph (road-like: low degree, wide weights), plain
        {"name": "rgg_1m_plain", "via": "device", "algorithm": "boruvka", "graph": "rgg2d",
         "n": 1000003, "degree": 16.0, "max_weight": W31, "threshold": 4},
        # an ordinary random graph of odd sizes
        {"name": "gnm_1m_filter", "via": "device", "algorithm": "filter_boruvka",
         "graph": "gnm", "n": 1000003, "m": 16000001, "max_weight": W8, "threshold": 4},
        # the three full-size benchmark graphs
        {"name": "gnm_2e24_filter", "via": "device", "algorithm": "filter_boruvka",
         "graph": "gnm", "n": 1 << 24, "m": 1 << 28, "max_weight": W8, "threshold": 4},
        {"name": "gnm_2e24_plain", "via": "device", "algorithm": "boruvka", "graph": "gnm",
         "n": 1 << 24, "m": 1 << 28, "max_weight": W8, "threshold": 4},
        {"name": "rgg_2e24_filter", "via": "device", "algorithm": "filter_boruvka",
         "graph": "rgg2d", "n": 1 << 24, "degree": 16.0, "max_weight": W31, "threshold": 4},
        {"name": "rhg_2e23_filter", "via": "device", "algorithm": "filter_boruvka",
         "graph": "rhg", "n": 1 << 23, "degree": 32.0, "max_weight": W8, "threshold": 4},
        # a burst of serving requests, n log-uniform in [2^8, 2^18], inputs in HBM
        {"name": "serve_512", "via": "server", "algorithm": "filter_boruvka", "graph": "gnm",
         "requests": 512, "max_weight": W8, "threshold": 4},
        # the drop-in call on host records (24 bytes each) with the defaults
        {"name": "gnm_2e17_host", "via": "host", "algorithm": "boruvka", "graph": "gnm",
         "n": 1 << 17, "m": 3 << 19, "max_weight": W8, "threshold": 4, "compression": 0},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    via = rng.choice(["device"] * 7 + ["noalloc", "server", "host"])
    algorithm = rng.choice(["boruvka", "filter_boruvka"])
    c = {"via": via, "algorithm": algorithm, "graph": "gnm",
         "max_weight": rng.choice([W8, W8, W31]), "threshold": rng.choice([4, 4, 4, 2, 3, 6])}
    if via == "server":
        c["requests"] = _log_uniform(rng, 1, 512)
        return c
    # most records a drawn case may have: the no-allocation entry's limit, a
    # host copy of about 100 MB, or a quarter of the headline graph
    most = {"device": 1 << 27, "noalloc": 1 << 20, "host": 1 << 22}[via]
    c["n"] = _log_uniform(rng, 256, min(most // (32 if via == "host" else 4), 1 << 24))
    # (host results have the forest's own length: dense enough to be connected)
    degree = _log_uniform(rng, 24 if via == "host" else 4, 64)
    degree = max(2, min(degree, most // c["n"], c["n"] // 4))
    c["graph"] = rng.choice(["gnm", "gnm", "rgg2d", "rhg"]) if via == "device" else "gnm"
    if c["graph"] == "gnm":
        c["m"] = max(1, c["n"] * degree // 2 - rng.randrange(1, 64))
    else:
        c["degree"] = float(min(degree, 32))
    if via == "host":
        c["compression"] = rng.choice([0, 1])
    return c


# ------------------------------------------------------------------ inputs
def _request_specs(case):
    """(n, undirected edges) of each request of a burst: the case's, whatever
    the seed of the graphs."""
    rng = np.random.default_rng(case["requests"])
    specs = []
    for _ in range(case["requests"]):
        n = int(round(2 ** rng.uniform(8, 18)))
        degree = rng.uniform(8, 32)
        specs.append((n, int(min(n * degree / 2, n * (n - 1) // 2))))
    return specs


def _graph_seed(seed):
    return (int(seed) * 0x9E3779B97F4A7C15 + 0x4B414D53) & ((1 << 63) - 1)


def _device_gnm(ctx, n, m, max_weight, seed, out=None):
    if out is None:
        out = torch.empty((3, 2 * m), dtype=torch.int32, device="cuda")
    ctx.gen_gnm_device(n, m, max_weight, seed, out[0], out[1], out[2])
    return [out[0], out[1], out[2]]


def _device_graph(case, seed):
    """(src, dst, weight) on the device, sorted and symmetric."""
    ctx = k.Context()   # its own: the generators' scratch goes with it
    try:
        s = _graph_seed(seed)
        if case["graph"] == "gnm":
            return _device_gnm(ctx, case["n"], case["m"], case["max_weight"], s)
        if case["graph"] == "rgg2d":
            return ctx.gen_rgg2d_device(case["n"], case["degree"], case["max_weight"], s)
        return ctx.gen_rhg_device(case["n"], case["degree"], 2.8, case["max_weight"], s)
    finally:
        ctx.close()


def _config(case):
    return k.AlgorithmConfig(compression=case.get("compression", 0),
                             filter_threshold=case["threshold"])


def _algorithm(case):
    return k.BORUVKA if case["algorithm"] == "boruvka" else k.FILTER_BORUVKA


def prepare(case, seed):
    st = {"via": case["via"], "algorithm": _algorithm(case), "config": _config(case)}
    if case["via"] == "server":
        specs = _request_specs(case)
        offs = np.concatenate([[0], np.cumsum([2 * m for _, m in specs])])
        pool = torch.empty((3, int(offs[-1])), dtype=torch.int32, device="cuda")
        first = np.concatenate([[0], np.cumsum([n for n, _ in specs])])
        st["out"] = torch.zeros((3, int(first[-1])), dtype=torch.int32, device="cuda")
        ctx = k.Context()
        reqs = []
        for i, (n, m) in enumerate(specs):
            part = pool[:, int(offs[i]):int(offs[i + 1])]
            _device_gnm(ctx, n, m, case["max_weight"], _graph_seed(seed) + i, part)
            out = st["out"][:, int(first[i]):int(first[i + 1])]
            reqs.append((part[0], part[1], part[2], n, (out[0], out[1], out[2])))
        ctx.close()
        torch.cuda.synchronize()
        st["requests"] = reqs
        st["server"] = k.Server(algorithm=st["algorithm"], filter_threshold=case["threshold"],
                                max_batch_records=max(int(offs[-1]), 1 << 20),
                                queue_capacity=len(reqs) + 16)
        return st
    arrays = _device_graph(case, seed)
    if case["via"] == "host":
        host = [a.cpu().numpy().view(np.uint32) for a in arrays]
        st["edges"] = k.to_wedges(*host)
        st["call"] = k.boruvka if case["algorithm"] == "boruvka" else k.filter_boruvka
        return st
    st["in"], st["n"], st["m"] = arrays, case["n"], int(arrays[0].numel())
    st["out"] = torch.zeros((3, case["n"]), dtype=torch.int32, device="cuda")
    if case["via"] == "device":
        st["context"] = k.Context()
        st["context"].reserve(st["m"], st["n"])
    torch.cuda.synchronize()
    return st


def run(st):
    if st["via"] == "server":
        srv = st["server"]
        tickets = [srv.submit(s, d, w, n, out=out) for s, d, w, n, out in st["requests"]]
        results = [srv.wait(t) for t in tickets]
        # every request's output arrays, with its count and weight
        return {"mst": st["out"],
                "count": np.array([r["mst_edges"] for r, _ in results], dtype=np.int64),
                "weight": np.array([r["total_weight"] for r, _ in results], dtype=np.int64)}
    if st["via"] == "host":
        mst, weight = st["call"](st["edges"], st["config"])
        return {"mst": [mst["src"], mst["dst"], mst["weight"]],
                "count": len(mst), "weight": weight}
    s, d, w = st["in"]
    os_, od, ow = st["out"]
    solve = k.solve_device_noalloc if st["via"] == "noalloc" else st["context"].solve_device
    count, weight = solve(s, d, w, st["m"], st["n"], os_, od, ow, st["n"],
                          algorithm=st["algorithm"], config=st["config"])
    return {"mst": st["out"], "count": count, "weight": weight}


def work(case):
    """Every record read once (12 bytes, 24 on the host), every MST edge
    written once; comparisons only, no floating-point work."""
    if case["via"] == "server":
        # expectation over the request sizes: n log-uniform in [2^8, 2^18],
        # degree U[8, 32]
        n = ((1 << 18) - (1 << 8)) / math.log(1 << 10)
        return {"bytes": case["requests"] * (12.0 * 20.0 * n + 12.0 * n), "flops": 0.0}
    records = 2 * case["m"] if case["graph"] == "gnm" else case["n"] * case["degree"]
    size = 24.0 if case["via"] == "host" else 12.0
    return {"bytes": size * (records + case["n"]), "flops": 0.0}


# ------------------------------------------------------------------- exact
def _forest(n, s, d, w):
    """The minimum spanning forest under the strict order (weight, min, max),
    by Boruvka rounds on edge ranks in numpy: (min, max, weight) sorted by
    (min, max)."""
    fwd = s < d
    s, d, w = (x[fwd].astype(np.int64) for x in (s, d, w))
    rank = np.empty(len(s), dtype=np.int64)
    order = np.lexsort((d, s, w))
    rank[order] = np.arange(len(s))
    comp = np.arange(n, dtype=np.int64)
    taken = np.zeros(len(s), dtype=bool)
    live = np.arange(len(s))
    while len(live):
        a, b = comp[s[live]], comp[d[live]]
        keep = a != b
        live, a, b = live[keep], a[keep], b[keep]
        if not len(live):
            break
        best = np.full(n, len(s), dtype=np.int64)
        np.minimum.at(best, a, rank[live])
        np.minimum.at(best, b, rank[live])
        roots = np.flatnonzero(best < len(s))
        e = order[best[roots]]
        taken[e] = True
        other = np.where(comp[s[e]] == roots, comp[d[e]], comp[s[e]])
        parent = np.arange(n, dtype=np.int64)
        parent[roots] = other
        mutual = (parent[parent] == np.arange(n)) & (np.arange(n) < parent)
        parent[mutual] = np.flatnonzero(mutual)
        while True:
            up = parent[parent]
            if np.array_equal(up, parent):
                break
            parent = up
        comp = parent[comp]
    e = np.flatnonzero(taken)
    e = e[np.lexsort((d[e], s[e]))]
    return s[e], d[e], w[e]


def _padded(forest, n):
    """The device output arrays: entries past the forest keep their zeros."""
    out = np.zeros((3, n), dtype=np.int32)
    out[:, :len(forest[0])] = np.stack(forest)
    return out


def exact(case, seed):
    if case["via"] == "server":
        specs = _request_specs(case)
        if sum(2 * m for _, m in specs) > EXACT_RECORDS:
            return None
        got = []
        for i, (n, m) in enumerate(specs):
            one = k.gen_gnm_host(n, m, case["max_weight"], _graph_seed(seed) + i)
            got.append(_forest(n, *one))
        return {"mst": np.concatenate([_padded(f, n) for f, (n, _) in zip(got, specs)], axis=1),
                "count": np.array([len(f[0]) for f in got], dtype=np.int64),
                "weight": np.array([int(f[2].sum()) for f in got], dtype=np.int64)}
    records = 2 * case["m"] if case["graph"] == "gnm" else case["n"] * case["degree"]
    if records > EXACT_RECORDS:
        return None
    s, d, w = (a.cpu().numpy().view(np.uint32) for a in _device_graph(case, seed))
    a, b, ww = _forest(case["n"], s, d, w)
    if case["via"] == "host":
        mst = [x.astype(t) for x, t in zip((a, b, ww), (np.uint64, np.uint64, np.uint32))]
    else:
        mst = _padded((a, b, ww), case["n"])
    return {"mst": mst, "count": len(a), "weight": int(ww.sum())}
