"""The host entry points stage their records through pinned chunks on several
threads: sizes at the chunks' edges, fewer and more chunks than slots, one
thread, and an id past 32 bits in any chunk."""
import numpy as np
import pytest

import kamsta_amd as k
import oracle

pytestmark = pytest.mark.gpu

CHUNK = 1 << 14  # records: the smallest chunk


def records(n, edges, seed):
    return k.to_wedges(*k.gen_gnm_host(n, edges, 254, seed))


def same(got, exp):
    return all(np.array_equal(got[f], exp[f]) for f in ("src", "dst", "weight"))


@pytest.mark.parametrize("threads", ["1", "3", "16"])
@pytest.mark.parametrize("n,edges", [
    (3, 2), (300, CHUNK // 2 - 1), (300, CHUNK // 2), (300, CHUNK // 2 + 1), (2000, CHUNK + 1),
    (60000, 8 * CHUNK), (60000, 8 * CHUNK + 1), (100000, (1 << 20) + 5), (200000, 1 << 21)])
def test_chunks(gpu, monkeypatch, threads, n, edges):
    monkeypatch.setenv("OMP_NUM_THREADS", threads)
    rec = records(n, edges, edges)
    exp, exp_w = oracle.kruskal(rec)
    got, got_w = k.boruvka(rec)
    assert got_w == exp_w and same(got, exp)


@pytest.mark.parametrize("field", ["src", "dst"])
@pytest.mark.parametrize("at", [0, CHUNK - 1, CHUNK, 5 * CHUNK + 7, -1])
def test_wide_id_refused(gpu, field, at):
    rec = records(5000, 4 * CHUNK, 3)
    good, good_w = k.boruvka(rec)
    for wide in (0xFFFFFFFF, 1 << 40):
        bad = rec.copy()
        bad[field][at] = wide
        with pytest.raises(k.KmstError) as e:
            k.boruvka(bad)
        assert e.value.status == k.KMST_EINVAL
    again, again_w = k.boruvka(rec)
    assert again_w == good_w and same(again, good)
