"""The two forms of the walk kernel at the partition count between them, and what
each append mode takes, against the CPU oracle bit for bit."""
import numpy as np
import pytest

import lighttraffic_amd as lt
from oracle import ffi as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("append_mode", [0, 1, 2])
@pytest.mark.parametrize("P", [1, 255, 256, 257, 1024, 1025])
def test_partition_counts(P, append_mode):
    """One vertex with four neighbours a partition; sources one at a time and in
    batches, 1, 2 and 4 walkers a thread, all slots or half of them."""
    print(f"walk forms P={P} append_mode={append_mode}", flush=True)
    rng = np.random.default_rng(P)
    g = lt.Graph.from_csr(4 * np.arange(P + 1, dtype=np.uint64), rng.integers(0, P, 4 * P).astype(np.uint32))
    part = lt.Partition.build(g, 32)
    assert part.count == P
    w, l = 9973, 5
    rc, re, _ = oracle.pagerank(g.rowptr(), g.col(), w, l, endpoints=True, threads=8)
    for wpt, span in ((1, "partition"), (2, "resident"), (4, "resident")):
        if P > 300 and span == "partition":
            continue  # a round a partition: long, and nothing new
        eng = lt.Engine(g, part, num_device_partitions=max(1, P // 2), span=span, walkers_per_thread=wpt,
                        resident_batch=16, zc_batch=16, append_mode=append_mode)
        counts, ends = eng.pagerank(w, l, endpoints=True)
        assert np.array_equal(counts, rc) and np.array_equal(ends, re)


@pytest.mark.parametrize("slots", [1, 3, 400])
@pytest.mark.parametrize("P", [1, 2, 255, 256, 257, 600])
def test_device_loop_partition_counts(P, slots):
    """The device's decisions with a partition a thread, one more, several; few
    slots (evictions), some, and one for each of most partitions."""
    print(f"device loop P={P} slots={slots}", flush=True)
    rng = np.random.default_rng(P)
    g = lt.Graph.from_csr(4 * np.arange(P + 1, dtype=np.uint64), rng.integers(0, P, 4 * P).astype(np.uint32))
    part = lt.Partition.build(g, 32)
    assert part.count == P
    w, l = 2503, 4
    rc, re, _ = oracle.pagerank(g.rowptr(), g.col(), w, l, endpoints=True, threads=8)
    for zc in (0, 5):
        eng = lt.Engine(g, part, num_device_partitions=min(slots, P), zerocopy_threshold=zc, device_schedule=1)
        for _ in range(2):
            counts, ends = eng.pagerank(w, l, endpoints=True)
            assert np.array_equal(counts, rc) and np.array_equal(ends, re)


@pytest.mark.parametrize("kw", [{}, {"zerocopy_threshold": 1 << 30, "zc_batch": 16}, {"pack_partitions": 2},
                                {"device_schedule": 1}], ids=["resident", "zerocopy", "blocks", "device"])
def test_partitions_within_a_lookup_step(kw):
    """131 075 vertices are looked up four at a time; the first 64 of them and the
    last fill a partition each."""
    print(f"lookup {kw}", flush=True)
    rng = np.random.default_rng(5)
    deg = np.ones(131075, np.uint64)
    deg[:64] = deg[-1] = 2000
    rowptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64)
    col = rng.integers(0, len(deg), int(rowptr[-1]))
    col[::3] %= 64
    g = lt.Graph.from_csr(rowptr, col.astype(np.uint32))
    part = lt.Partition.build(g, 8100)
    assert part.count > 200
    w, l = 30011, 6
    rc, re, _ = oracle.pagerank(g.rowptr(), g.col(), w, l, endpoints=True, threads=8)
    eng = lt.Engine(g, part, num_device_partitions=part.count // 2, span="resident",
                    **{"zerocopy_threshold": 100, "resident_batch": 16, **kw})
    counts, ends = eng.pagerank(w, l, endpoints=True)
    assert np.array_equal(counts, rc) and np.array_equal(ends, re)


@pytest.mark.parametrize("depth", [1, 2, 3, 8])
def test_table_entries_told_to_the_walk(depth):
    """Loads ahead change up to two entries each between launches: as many as a walk
    is told of, one more, and many."""
    print(f"table entries depth={depth}", flush=True)
    g = lt.Graph.rmat(15, 16)
    part = lt.Partition.build(g, 32 << 10)
    w, l = 40009, 8
    rc, re, _ = oracle.pagerank(g.rowptr(), g.col(), w, l, endpoints=True, threads=8)
    eng = lt.Engine(g, part, num_device_partitions=part.count // 2, span="resident", policy="learned",
                    prefetch_plain=1, prefetch_depth=depth, zerocopy_threshold=50, resident_batch=16)
    for _ in range(2):
        counts, ends = eng.pagerank(w, l, endpoints=True)
        assert np.array_equal(counts, rc) and np.array_equal(ends, re)
    assert eng.stats()["prefetch_issued"] > 0
