"""Visit counting through the visit log (jobs of many visits) against the CPU
oracle bit for bit: one bin of vertices, a few, many; logs counted once, in
pieces, and overfull; flat jobs, the host's queues and the device loop."""
import numpy as np
import pytest

import lighttraffic_amd as lt
from oracle import ffi as oracle

pytestmark = pytest.mark.gpu


def _ring(V):
    """V vertices with 1-4 random neighbours each."""
    rng = np.random.default_rng(V)
    rowptr = np.concatenate([[0], np.cumsum(rng.integers(1, 5, V))]).astype(np.uint64)
    return lt.Graph.from_csr(rowptr, rng.integers(0, V, int(rowptr[-1])).astype(np.uint32))


def _check(g, eng, w, l):
    counts, ends = eng.pagerank(w, l, endpoints=True)
    rc, re, _ = oracle.pagerank(g.rowptr(), g.col(), w, l, endpoints=True, threads=16)
    assert np.array_equal(counts, rc) and np.array_equal(ends, re)


@pytest.mark.parametrize("V", [1, 32768, 32769, 65536, 131072, 131073, 500001])
def test_flat_jobs(V):
    """Visits around the log's smallest job, whole and partial tiles, V at the bins' edges."""
    print(f"visit log flat V={V}", flush=True)
    g = _ring(V)
    eng = lt.Engine(g, lt.Partition.build(g, 64 << 20), zerocopy_threshold=0)
    eng.pagerank(1000, 2)
    for w, l in ((262143, 1), (262144, 1), (16384 * 16 + 1, 2), (123457, 10)):
        _check(g, eng, w, l)
    for w in (262143, 300000):
        counts = eng.ppr(w, source=V - 1)
        assert np.array_equal(counts, oracle.ppr(g.rowptr(), g.col(), w, source=V - 1, threads=16)[0])


@pytest.mark.parametrize("V", [1, 32768, 32769, 65536, 131072, 131073, 500001])
def test_flat_jobs_of_an_engine_with_a_log(V):
    """The same behind a job of 34 M visits, which allocates the log that they use."""
    print(f"visit log kept V={V}", flush=True)
    g = _ring(V)
    eng = lt.Engine(g, lt.Partition.build(g, 64 << 20), zerocopy_threshold=0)
    _check(g, eng, 1 << 20, 32)
    for w, l in ((262143, 1), (262144, 1), (16384 * 16 + 1, 2), (123457, 10)):
        _check(g, eng, w, l)
    for w in (262143, 300000):
        counts = eng.ppr(w, source=V - 1)
        assert np.array_equal(counts, oracle.ppr(g.rowptr(), g.col(), w, source=V - 1, threads=16)[0])


def test_flat_job_in_pieces():
    """75 M visits: more than one log holds."""
    print("visit log pieces", flush=True)
    g = lt.Graph.rmat(17, 8)
    eng = lt.Engine(g, lt.Partition.build(g, 64 << 20), zerocopy_threshold=0)
    eng.pagerank(1000, 2)
    _check(g, eng, 750001, 100)


@pytest.mark.parametrize("kw", [{"span": "resident", "resident_batch": 16, "walkers_per_thread": 4},
                                {"span": "partition", "pack_partitions": 2},
                                {"span": "resident", "device_schedule": 1},
                                {"num_device_walkers": 200000}], ids=["batches", "partition", "device", "spill"])
@pytest.mark.parametrize("w,l", [(900001, 20), (750001, 100)])
def test_queued_jobs(kw, w, l):
    """18 M visits in one log; 75 M: the log is counted as it fills, and what a
    launch visits beyond it is counted directly."""
    print(f"visit log queued {kw} w={w} l={l}", flush=True)
    g = lt.Graph.rmat(18, 8)
    part = lt.Partition.build(g, 1 << 20)
    eng = lt.Engine(g, part, **{"num_device_partitions": part.count // 2, **kw})
    _check(g, eng, w, l)
    _check(g, eng, w - 1, l)
