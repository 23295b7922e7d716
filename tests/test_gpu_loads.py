"""Partition loads by one kernel and by DMA, slices at both sides of the line
between them, against the CPU oracle bit for bit."""
import numpy as np
import pytest

import lighttraffic_amd as lt
from oracle import ffi as oracle

pytestmark = pytest.mark.gpu

_LINE = 1280 << 10  # bytes of a partition's two slices
_LINE_ONE = 256 << 10


@pytest.mark.parametrize("mode", ["plain", "ahead", "device"])
@pytest.mark.parametrize("over", [-4, 0, 4, _LINE - 12])
def test_slices_around_the_line(over, mode):
    """Five partitions of one vertex and its edges each, four of them with slices
    of the line's bytes, a word or an edge less or more, and of about twice that."""
    _slices(_LINE, over, mode)


@pytest.mark.parametrize("over", [-4, 0, 4, _LINE_ONE - 12])
def test_slices_around_the_line_of_walks_in_one_partition(over):
    _slices(_LINE_ONE, over, "plain")


def _slices(line, over, mode):
    print(f"loads {mode} line={line} over={over}", flush=True)
    deg = (line + over - 16) // 4
    degs = np.array([deg, deg, 7, deg - 1, deg], np.uint64)
    rng = np.random.default_rng(deg)
    rowptr = np.concatenate([[0], np.cumsum(degs)]).astype(np.uint64)
    col = rng.integers(0, 5, int(rowptr[-1])).astype(np.uint32)
    g = lt.Graph.from_csr(rowptr, col)
    part = lt.Partition.build(g, deg * 4 + 32)
    assert part.count >= 4
    kw = {"plain": {}, "ahead": {"policy": "learned", "prefetch_plain": 1, "prefetch_depth": 2, "span": "resident"},
          "device": {"device_schedule": 1}}[mode]
    eng = lt.Engine(g, part, num_device_partitions=3, zerocopy_threshold=0, pack_partitions=0, **kw)
    for _ in range(2):
        counts, ends = eng.pagerank(20001, 9, endpoints=True)
        rc, re, _ = oracle.pagerank(g.rowptr(), g.col(), 20001, 9, endpoints=True, threads=8)
        assert np.array_equal(counts, rc) and np.array_equal(ends, re)
    assert eng.stats()["graph_loading_calls"] > 3
