"""running_ms is the host's time, by whichever route a job walks: jobs of both
routes are compared by it, and a device clock read as 32 bits of 10 ns wraps
after 42.9 s."""
import time

import pytest

import lighttraffic_amd as lt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [{"zerocopy_threshold": 0}, {"num_device_partitions": 3, "span": "resident"}],
                         ids=["flat", "queues"])
@pytest.mark.parametrize("w", [1000, 100000, 1200000])
def test_running_time_is_the_hosts(kw, w):
    """Results by each way to the host: the last kernels, copies, the ring and the
    walk itself.  A clock of whole 10 ns ticks would give multiples of 10 ns in
    all 24 jobs; the host's clock does by chance once in 10^24."""
    print(f"running time w={w} {kw}", flush=True)
    g = lt.Graph.rmat(13, 8)
    eng = lt.Engine(g, lt.Partition.build(g, 32 << 20 if "span" not in kw else 32 << 10), **kw)
    ns = []
    for job in range(24):
        t = time.perf_counter()
        if job % 2:
            eng.genericwalk(w, 3, moves=True)
        else:
            eng.pagerank(w, 3, endpoints=True)
        call = (time.perf_counter() - t) * 1e9
        ns.append(round(eng.stats()["running_ms"] * 1e6))
        assert 0 < ns[-1] <= call
    assert any(x % 10 for x in ns), ns
