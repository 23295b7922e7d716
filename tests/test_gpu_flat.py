"""Jobs on a graph that lies whole in HBM (every partition cached, span
resident with batches, or one partition), which are walked over the flat
arrays in one launch, against the CPU oracle bit for bit."""
import numpy as np
import pytest

import lighttraffic_amd as lt
from oracle import ffi as oracle

pytestmark = pytest.mark.gpu


def _dead_end_graph():
    """Rows of 0-5 edges, the last vertices without any."""
    rng = np.random.default_rng(3)
    V = 1500
    deg = rng.integers(0, 6, V)
    deg[-40:] = 0
    rowptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64)
    return lt.Graph.from_csr(rowptr, rng.integers(0, V, int(rowptr[-1])).astype(np.uint32))


@pytest.fixture(scope="module", params=["rmat", "dead-ends", "rmat16"])
def graph(request):
    return {"rmat": lambda: lt.Graph.rmat(12, 8), "dead-ends": _dead_end_graph,
            "rmat16": lambda: lt.Graph.rmat(16, 8)}[request.param]()


@pytest.mark.parametrize("pbytes,kw", [(32 << 20, {}), (16 << 10, {"span": "resident", "resident_batch": 16}),
                                       (16 << 10, {"span": "resident", "resident_batch": 16, "pack_partitions": 1})],
                         ids=["one-partition", "many", "many-unpacked"])
@pytest.mark.parametrize("w", [1, 256, 257, 70001])
def test_flat_walks_match_the_oracle(graph, pbytes, kw, w):
    print(f"flat V={graph.num_node} {pbytes} {kw} w={w}", flush=True)
    part = lt.Partition.build(graph, max(pbytes, int(np.diff(graph.rowptr()).max()) * 4 + 64))
    rp, col = graph.rowptr(), graph.col()
    eng = lt.Engine(graph, part, zerocopy_threshold=0, **kw)
    for _ in range(3):  # fill the cache: a partition is loaded when a walker first reaches it
        eng.genericwalk(50000, 12)

    def flat():
        st = eng.stats()
        assert st["iterations"] == 1 and st["kernel_launches"] == 1 and st["graph_loading_calls"] == 0
        return st

    for l in (0, 1, 9):
        counts, ends = eng.pagerank(w, l, endpoints=True)
        rc, re, rst = oracle.pagerank(rp, col, w, l, endpoints=True)
        st = flat()
        assert np.array_equal(counts, rc) and np.array_equal(ends, re)
        assert (st["moves"], st["teleports"], st["visits"]) == (rst[0], rst[1], rst[2])
        assert st["residencies"] == (w if l else 0)
        ends, moves = eng.genericwalk(w, l, runs=2, moves=True)
        re, rm, _ = oracle.genericwalk(rp, col, w, l, runs=2)
        assert np.array_equal(ends, re) and np.array_equal(moves, rm)
        assert flat()["moves"] == int(rm.sum())
        assert np.array_equal(eng.genericwalk_paths(w, l), oracle.genericwalk_paths(rp, col, w, l))
    for src in (0, graph.num_node - 1):
        counts, ends = eng.ppr(w, source=src, prob=0.15, endpoints=True)
        rc, re, rst = oracle.ppr(rp, col, w, source=src, prob=0.15, endpoints=True)
        assert np.array_equal(counts, rc) and np.array_equal(ends, re)
        assert flat()["moves"] == rst[0]
    sources = np.random.default_rng(1).integers(0, graph.num_node, 9).astype(np.uint32)
    qc = np.array([1, 0, w, 3, 0, 0, 2 * w + 5, 1, 0], np.uint64)
    assert np.array_equal(eng.ppr_batch(sources, qc), oracle.ppr_batch(rp, col, sources, qc)[0])
    flat()
