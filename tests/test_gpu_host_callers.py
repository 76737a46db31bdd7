"""Several callers of the host entry points: what a call does to its own records
does not wait for another caller's solve."""
import threading
import time

import numpy as np
import pytest

import kamsta_amd as k

pytestmark = pytest.mark.gpu


def test_coded_records_are_converted_beside_another_call(gpu):
    """A wide id in a difference-coded call is met while the records are
    converted: the call ends long before the large one that began before it."""
    rec = k.to_wedges(*k.gen_gnm_host(1 << 20, 1 << 23, 254, 3))
    bad = rec[:3].copy()
    bad["dst"][1] = 1 << 40
    k.boruvka(rec)  # workspaces and staging are there
    with pytest.raises(k.KmstError):
        k.boruvka(bad, k.AlgorithmConfig(compression=1))  # a first throw takes 85 ms
    took = {}

    def large():
        began.set()
        t = time.perf_counter()
        k.boruvka(rec)
        took["large"] = time.perf_counter() - t

    began = threading.Event()
    other = threading.Thread(target=large)
    other.start()
    began.wait(30)
    time.sleep(0.002)
    t = time.perf_counter()
    with pytest.raises(k.KmstError) as e:
        k.boruvka(bad, k.AlgorithmConfig(compression=1))
    took["refused"] = time.perf_counter() - t
    other.join(60)
    assert e.value.status == k.KMST_EINVAL
    assert took["refused"] < took["large"] / 10, took
