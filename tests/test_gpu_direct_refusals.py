"""What the direct solve (kmst_union.hip) leaves behind where it ends without a
forest: the caller's arrays as they were, and a context that goes on."""
import dataclasses

import numpy as np
import pytest

import kamsta_amd as k

pytestmark = pytest.mark.gpu


def dev(torch, x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.uint32).view(np.int32)).cuda()


# one workgroup in LDS; one and several workgroups of the general solve
@pytest.mark.parametrize("n,edges", [(200, 500), (4000, 9000), (4000, 40000)])
@pytest.mark.parametrize("short", [1, 1000, None])
def test_too_small_capacity_leaves_the_arrays(gpu, ctx, n, edges, short):
    """As the round loop does: nothing is written before the call is refused."""
    arrs = [dev(gpu, x) for x in k.gen_gnm_host(n, edges, 254, 5)]
    full = gpu.zeros((3, n), dtype=gpu.int32, device="cuda")
    cnt, _ = ctx.solve_device(*arrs, 2 * edges, n, *full, n)
    cap = 0 if short is None else max(cnt - short, 0)
    entry = ctx.get_tuning()
    for limit in (entry.persistent_max, 0):  # 0: the round loop
        try:
            ctx.set_tuning(dataclasses.replace(entry, persistent_max=limit))
            out = gpu.full((3, n), 77, dtype=gpu.int32, device="cuda")
            gpu.cuda.synchronize()
            with pytest.raises(k.KmstError) as e:
                ctx.solve_device(*arrs, 2 * edges, n, *out, cap)
            assert e.value.status == k.KMST_EINVAL
            assert bool((out == 77).all()), limit
        finally:
            ctx.set_tuning(entry)
    out = gpu.zeros((3, n), dtype=gpu.int32, device="cuda")
    gpu.cuda.synchronize()
    assert ctx.solve_device(*arrs, 2 * edges, n, *out, cnt)[0] == cnt
    assert gpu.equal(out, full)
