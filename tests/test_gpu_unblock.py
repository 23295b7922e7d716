"""Block images that only travel: with raw slots asked for all partitions the
columns are kept raw and jobs walk flat.  Against the CPU oracle bit for bit."""
import numpy as np
import pytest

import lighttraffic_amd as lt
from oracle import ffi as oracle

pytestmark = pytest.mark.gpu


def _graph(V, seed):
    """Degrees from 0 on: blocks of 16 edges with remainders, empty rows and,
    among the partitions, some that do not get smaller as blocks."""
    rng = np.random.default_rng(seed)
    deg = rng.integers(0, 40, V)
    deg[rng.integers(0, V, V // 4)] = 0
    rowptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64)
    col = rng.integers(0, V, int(rowptr[-1]))
    near = rng.random(len(col)) < 0.8  # most neighbours near: narrow blocks
    at = np.repeat(np.arange(V), deg)
    col = np.where(near & (at > V // 5), (at + col % 50) % V, col)
    return lt.Graph.from_csr(rowptr, col.astype(np.uint32))


@pytest.mark.parametrize("V", [17, 1000, 30011])
@pytest.mark.parametrize("slots", [0, "all", "less"])
def test_jobs(V, slots):
    print(f"unblock V={V} slots={slots}", flush=True)
    g = _graph(V, V)
    part = lt.Partition.build(g, max(1024, g.num_edge * 4 // 12))
    P = part.count
    n = {0: 0, "all": P, "less": max(1, P // 3)}[slots]
    eng = lt.Engine(g, part, num_device_partitions=n, pack_partitions=2, span="resident", resident_batch=16)
    with pytest.raises(lt.LTError):
        eng.fetch_partition(0, part.node_offsets(), part.edge_offsets())
    w = max(5000, P * 4200)
    rc, re, _ = oracle.pagerank(g.rowptr(), g.col(), w, 6, endpoints=True, threads=8)
    pc = oracle.ppr(g.rowptr(), g.col(), w, source=V - 2, threads=8)[0]
    for _ in range(2):
        counts, ends = eng.pagerank(w, 6, endpoints=True)
        assert np.array_equal(counts, rc) and np.array_equal(ends, re)
        assert np.array_equal(eng.ppr(w, source=V - 2), pc)
    if slots != "less":
        assert eng.stats()["iterations"] == 1 and eng.stats()["graph_loading_calls"] == 0


@pytest.mark.parametrize("slots", [0, 2])
def test_refused_fetch_says_why(slots):
    """With slots for all the columns are raw, so the reason is the copies' form."""
    g = _graph(1000, 5)
    eng = lt.Engine(g, lt.Partition.build(g, max(1024, g.num_edge * 4 // 6)), num_device_partitions=slots,
                    pack_partitions=2)
    with pytest.raises(lt.LTError, match="copies are block images"):
        eng.fetch_partition(0, eng.partition.node_offsets(), eng.partition.edge_offsets())
