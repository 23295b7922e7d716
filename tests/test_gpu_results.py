"""Results of every size on their way to the host (written by the job's last
kernels, through the ring of pinned buffers, or into it by the walk), against
the CPU oracle bit for bit; flat jobs and jobs through the queues."""
import numpy as np
import pytest

import lighttraffic_amd as lt
from oracle import ffi as oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def graph():
    return lt.Graph.rmat(14, 8)


@pytest.mark.parametrize("kw", [{"zerocopy_threshold": 0}, {"num_device_partitions": 3, "span": "resident"}],
                         ids=["flat", "queues"])
@pytest.mark.parametrize("w", [65536, 65537, 524288, 1048577, 3 * 1048576 + 77])
def test_results_by_walker(graph, kw, w):
    print(f"results w={w} {kw}", flush=True)
    rp, col = graph.rowptr(), graph.col()
    part = lt.Partition.build(graph, 32 << 20 if "span" not in kw else 64 << 10)
    eng = lt.Engine(graph, part, **kw)
    eng.genericwalk(10000, 3)
    re, rm, _ = oracle.genericwalk(rp, col, w, 4, threads=16)
    ends, moves = eng.genericwalk(w, 4, moves=True)
    assert np.array_equal(ends, re) and np.array_equal(moves, rm)
    assert np.array_equal(eng.genericwalk(w, 4)[0], re)
    assert np.array_equal(eng.genericwalk(w, 4, endpoints=False, moves=True)[1], rm)
    counts, ends = eng.ppr(w, source=3, endpoints=True)
    rc, re, _ = oracle.ppr(rp, col, w, source=3, endpoints=True, threads=16)
    assert np.array_equal(counts, rc) and np.array_equal(ends, re)
    counts, ends = eng.pagerank(w, 2, endpoints=True)
    rc, re, _ = oracle.pagerank(rp, col, w, 2, endpoints=True, threads=16)
    assert np.array_equal(counts, rc) and np.array_equal(ends, re)
    if w < 600000:
        assert np.array_equal(eng.genericwalk_paths(w, 4), oracle.genericwalk_paths(rp, col, w, 4))


@pytest.mark.parametrize("w", [70001, 524288, 1048577, 3 * 1048576 + 77])
def test_later_jobs_of_one_engine(graph, w):
    """The first large results go by plain copies, later ones through a ring that
    grows with them; both arrays of a flat walk are written into it in launches."""
    print(f"results of later jobs w={w}", flush=True)
    rp, col = graph.rowptr(), graph.col()
    eng = lt.Engine(graph, lt.Partition.build(graph, 32 << 20), zerocopy_threshold=0)
    for n in (66000, 66001, w, 70000, w):
        re, rm, _ = oracle.genericwalk(rp, col, n, 4, threads=16)
        ends, moves = eng.genericwalk(n, 4, moves=True)
        assert np.array_equal(ends, re) and np.array_equal(moves, rm)


@pytest.mark.parametrize("first", [66000, 1 << 20], ids=["small-ring", "large-ring"])
@pytest.mark.parametrize("w", [(1 << 19) - 1, 1 << 19, (1 << 20) - 1, 1 << 20, (1 << 20) + 1, 2097152 + 5])
def test_results_at_the_rings_edges(graph, w, first):
    """One array and two, around the sizes from which threads help and walks write the
    large ring, which a first job of many results gets with its loads; in the small
    one, after small results and before."""
    print(f"results at the rings' edges w={w} first={first}", flush=True)
    rp, col = graph.rowptr(), graph.col()
    eng = lt.Engine(graph, lt.Partition.build(graph, 32 << 20), zerocopy_threshold=0)
    for n in (first, w, 131072 + 1, w, 2 * w):
        re, rm, _ = oracle.genericwalk(rp, col, n, 4, threads=16)
        ends, moves = eng.genericwalk(n, 4, moves=True)
        assert np.array_equal(ends, re) and np.array_equal(moves, rm)
        assert np.array_equal(eng.genericwalk(n, 4)[0], re)
        assert np.array_equal(eng.genericwalk(n, 4, endpoints=False, moves=True)[1], rm)


def test_results_while_the_large_ring_gets_ready(graph):
    """Short jobs whose helpers read a part of the large ring each, until it is used."""
    print("results while the large ring gets ready", flush=True)
    rp, col = graph.rowptr(), graph.col()
    eng = lt.Engine(graph, lt.Partition.build(graph, 32 << 20), zerocopy_threshold=0)
    eng.genericwalk(1000, 2)
    re, rm, _ = oracle.genericwalk(rp, col, 1100003, 3, threads=16)
    rc, pe, _ = oracle.pagerank(rp, col, 1100003, 2, endpoints=True, threads=16)
    for job in range(30):
        if job % 3 == 2:
            counts, ends = eng.pagerank(1100003, 2, endpoints=True)
            assert np.array_equal(counts, rc) and np.array_equal(ends, pe), job
        else:
            ends, moves = eng.genericwalk(1100003, 3, moves=job % 3 == 1)
            assert np.array_equal(ends, re) and (moves is None or np.array_equal(moves, rm)), job
