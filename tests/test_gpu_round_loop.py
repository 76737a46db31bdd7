"""The round loop, which solves sparse inputs and what the direct solve calls
off: the tests of its kernels again, on contexts whose persistent-round limit is
one record off its default, so that no solve is direct."""
import dataclasses
import functools

import numpy as np
import pytest

import kamsta_amd as k
from test_gpu_output_order import (test_hubs_in_a_random_graph, test_hyperbolic_hubs,
                                   test_positional_geometric)
from test_gpu_parity import (test_contract_errors, test_contract_errors_with_weight_classes,
                             test_device_solve_and_stats, test_device_solve_misaligned_inputs,
                             test_gnm_vs_oracle, test_positional_multigraph,
                             test_rgg2d_positional_keys, test_rhg_hubs,
                             test_twin_relabels_on_a_random_graph)
from test_gpu_serving import (test_bad_request_does_not_poison_batch, test_batch_of_mixed_upload_forms,
                              test_batched_equals_alone_and_oracle, test_batched_wide_weights)
from test_gpu_tuning import gnm, test_every_tuning_gives_the_oracle_mst

pytestmark = pytest.mark.gpu

DEFAULT = k.Tuning()
OFF = dataclasses.replace(DEFAULT, persistent_max=DEFAULT.persistent_max - 1)


class RoundLoop(k.Context):
    def __init__(self):
        super().__init__(0)
        self.set_tuning(DEFAULT)

    def set_tuning(self, t):
        """What asks for the default limit gets the one beside it."""
        super().set_tuning(OFF if t == DEFAULT else dataclasses.replace(
            t, persistent_max=min(t.persistent_max, OFF.persistent_max)))

    def get_tuning(self):
        return dataclasses.replace(super().get_tuning(), persistent_max=DEFAULT.persistent_max)

    def solve_device(self, *args, **kw):
        result = super().solve_device(*args, **kw)
        assert not any(r["direct"] or r["chains"] for r in self.stats()["rounds"])
        return result


@pytest.fixture(scope="module")
def ctx(gpu):
    c = RoundLoop()
    yield c
    c.close()


@pytest.fixture(autouse=True)
def entries(gpu, ctx, monkeypatch):
    """The host entry points and the server on that tuning."""
    def solve(algorithm, edges, config=None):
        n = int(max(edges["src"].max(), edges["dst"].max())) + 1 if len(edges) else 0
        arrs = [gpu.from_numpy(edges[f].astype(np.uint32).view(np.int32)).cuda()
                for f in ("src", "dst", "weight")]
        out = gpu.empty((3, max(n, 1)), dtype=gpu.int32, device="cuda")
        gpu.cuda.synchronize()
        cnt, total = ctx.solve_device(*arrs, len(edges), n, *out, max(n, 1), algorithm=algorithm,
                                      config=config)
        return k.to_wedges(*(x[:cnt].cpu().numpy().view(np.uint32) for x in out)), total

    monkeypatch.setattr(k, "boruvka", functools.partial(solve, k.BORUVKA))
    monkeypatch.setattr(k, "filter_boruvka", functools.partial(solve, k.FILTER_BORUVKA))
    for f, name in ((k.boruvka, "boruvka"), (k.filter_boruvka, "filter_boruvka")):
        f.__name__ = name
    monkeypatch.setattr(k, "Server", functools.partial(k.Server, tuning=OFF))
