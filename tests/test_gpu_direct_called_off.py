"""A direct solve whose workgroups are not resident together is called off at its
first barrier: the round loop solves or refuses the call, and the next solve on
the context is direct again."""
import numpy as np
import pytest

import kamsta_amd as k
import oracle

pytestmark = pytest.mark.gpu


def dev(torch, x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.uint32).view(np.int32)).cuda()


def solve(torch, ctx, arrs, m, n, algo, cap=None):
    out = torch.full((3, n), 77, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    try:
        cnt, total = ctx.solve_device(*arrs, m, n, *out, n if cap is None else cap, algorithm=algo)
    except k.KmstError as e:
        return e.status, out.cpu().numpy().view(np.uint32), ctx.stats()
    return (cnt, total), out.cpu().numpy().view(np.uint32), ctx.stats()


@pytest.mark.parametrize("copy", ["0", "1"])
@pytest.mark.parametrize("n,edges,mw", [(4000, 40000, 254), (70000, 300000, (1 << 31) - 1),
                                        (1 << 18, 1 << 20, 254)])
def test_called_off(gpu, monkeypatch, copy, n, edges, mw):
    monkeypatch.setenv("KMST_READBACK_COPY", copy)
    ctx = k.Context()
    s, d, w = k.gen_gnm_host(n, edges, mw, 8)
    exp, exp_w = oracle.kruskal(k.to_wedges(s, d, w))
    arrs = [dev(gpu, x) for x in (s, d, w)]
    wrong = w.copy()
    wrong[5] += 1
    for algo in (k.BORUVKA, k.FILTER_BORUVKA):
        for off in (True, False, True, False):
            if off:
                ctx.call_off()
            got, out, st = solve(gpu, ctx, arrs, 2 * edges, n, algo)
            assert got == (len(exp), exp_w)
            for row, f in zip(out, ("src", "dst", "weight")):
                assert np.array_equal(row[:len(exp)], exp[f])
                assert (row[len(exp):] == 77).all()
            assert st["called_off"] == off
            assert any(r["direct"] for r in st["rounds"]) == (not off)
        ctx.call_off()
        got, out, st = solve(gpu, ctx, arrs, 2 * edges, n, algo, cap=len(exp) - 1)
        assert got == k.KMST_EINVAL and (out == 77).all() and st["called_off"]
        ctx.call_off()
        got, out, st = solve(gpu, ctx, arrs[:2] + [dev(gpu, wrong)], 2 * edges, n, algo)
        assert got == k.KMST_EASYMMETRIC and (out == 77).all() and st["called_off"]
    ctx.close()


def test_one_workgroup_has_no_one_to_wait_for(gpu):
    """A solve in one workgroup is not called off: the next larger one is."""
    ctx = k.Context()
    ctx.call_off()
    for n, edges, off in (200, 500, False), (4000, 40000, True), (4000, 40000, False):
        s, d, w = k.gen_gnm_host(n, edges, 254, 9)
        exp, exp_w = oracle.kruskal(k.to_wedges(s, d, w))
        got, _, st = solve(gpu, ctx, [dev(gpu, x) for x in (s, d, w)], 2 * edges, n, k.BORUVKA)
        assert got == (len(exp), exp_w) and st["called_off"] == off
    ctx.close()
