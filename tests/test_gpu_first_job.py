"""A new engine's first job: partitions loaded up front and walked flat, at both
sides of the rule, against the CPU oracle bit for bit."""
import numpy as np
import pytest

import lighttraffic_amd as lt
from oracle import ffi as oracle

pytestmark = pytest.mark.gpu


def _check(g, eng, w, l, flat):
    """First job by the expected route, second one flat, the same results."""
    rc, re, _ = oracle.pagerank(g.rowptr(), g.col(), w, l, endpoints=True, threads=8)
    for first in (True, False):
        counts, ends = eng.pagerank(w, l, endpoints=True)
        assert np.array_equal(counts, rc) and np.array_equal(ends, re)
        st = eng.stats()
        if first:
            assert (st["iterations"] == 1 and st["graph_loading_calls"] == eng.partition.count) == flat
            bytes_ = 8 * (g.num_node + eng.partition.count) + 4 * g.num_edge
            assert not flat or 0 < st["h2d_bytes_unpacked"] <= bytes_


@pytest.mark.parametrize("pack", [0, 1])
@pytest.mark.parametrize("rp", [0, 1])
@pytest.mark.parametrize("over", [-1, 0])
def test_several_partitions(over, rp, pack):
    print(f"first job over={over} rp={rp} pack={pack}", flush=True)
    g = lt.Graph.rmat(13, 16)
    part = lt.Partition.build(g, 32 << 10)
    assert part.count > 4
    eng = lt.Engine(g, part, span="resident", resident_batch=16, zerocopy_threshold=0, rowptr_resident=rp,
                    pack_partitions=pack)
    _check(g, eng, part.count * 4096 + over, 3, over >= 0)


@pytest.mark.parametrize("w,zc", [(1, 1), (99, 100), (100, 100), (4097, 0)])
def test_one_partition(w, zc):
    """One partition: loaded at once unless it is read in place."""
    print(f"first job w={w} zc={zc}", flush=True)
    g = lt.Graph.rmat(10, 8)
    part = lt.Partition.build(g, 64 << 20)
    assert part.count == 1
    eng = lt.Engine(g, part, zerocopy_threshold=zc)
    rc, re, _ = oracle.pagerank(g.rowptr(), g.col(), w, 5, endpoints=True, threads=8)
    for job in range(2):
        counts, ends = eng.pagerank(w, 5, endpoints=True)
        assert np.array_equal(counts, rc) and np.array_equal(ends, re)
        st = eng.stats()
        assert st["graph_loading_calls"] == (1 if job == 0 and w >= zc else 0)
        assert st["zerocopy_calls"] == (0 if w >= zc else 1)


def test_some_partitions_cached_and_ppr():
    """Walkers of one source load what they reach; the next job loads the rest."""
    print("first job ppr, then pagerank", flush=True)
    g = lt.Graph.rmat(13, 16)
    part = lt.Partition.build(g, 32 << 10)
    eng = lt.Engine(g, part, span="resident", resident_batch=16, zerocopy_threshold=2000)
    w = 3000
    assert np.array_equal(eng.ppr(w, source=5), oracle.ppr(g.rowptr(), g.col(), w, source=5, threads=8)[0])
    loaded = eng.stats()["graph_loading_calls"]
    assert 0 < loaded < part.count
    w = part.count * 4096
    rc, re, _ = oracle.pagerank(g.rowptr(), g.col(), w, 3, endpoints=True, threads=8)
    counts, ends = eng.pagerank(w, 3, endpoints=True)
    assert np.array_equal(counts, rc) and np.array_equal(ends, re)
    assert eng.stats()["graph_loading_calls"] == part.count - loaded


@pytest.mark.parametrize("few", [1, 0])
def test_batched_ppr(few):
    """As many sources as partitions load them all at once; with one less, the
    queues load them."""
    print(f"first job batched ppr few={few}", flush=True)
    g = lt.Graph.rmat(14, 16)
    part = lt.Partition.build(g, 64 << 10)
    P = part.count
    nq = P - few
    assert nq > P // 8
    eng = lt.Engine(g, part, span="resident", resident_batch=16, zerocopy_threshold=0)
    src = np.arange(nq, dtype=np.uint32) * 7
    cnt = np.full(nq, -(-P * 4096 // nq), np.uint64)
    re, _ = oracle.ppr_batch(g.rowptr(), g.col(), src, cnt, threads=8)
    for first in (True, False):
        assert np.array_equal(eng.ppr_batch(src, cnt), re)
        st = eng.stats()
        if first:
            assert (st["iterations"] == 1 and st["graph_loading_calls"] == P) == (few == 0)
