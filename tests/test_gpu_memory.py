"""Jobs whose allocations fail, forced from the host (hipfail/): no failed one
leaves an engine that later jobs cannot use.  Each child process makes the
chosen runtime calls fail and checks its jobs against the CPU oracle."""
import ctypes
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
MALLOC, HOST_MALLOC, MEMCPY_ASYNC = range(3)

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("hipfail") / "libhipfail.so")
    subprocess.run(["gcc", "-O1", "-fPIC", "-shared", "-o", path, os.path.join(HERE, "hipfail", "hipfail.c"), "-ldl"],
                   check=True)
    return path


def child(shim, *args):
    print("memory", *args, flush=True)
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__), shim, *map(str, args)], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("done\n"), r.stdout[-2000:] + r.stderr[-2000:]


@pytest.mark.parametrize("form", ["flat", "queues", "spill", "batch", "device"])
def test_after_a_failed_allocation(shim, form):
    """Every device allocation of a job fails in turn, after a smaller job had run."""
    child(shim, "after", form)


@pytest.mark.parametrize("what", ["log", "kept_log", "offsets"])
def test_what_only_speeds_a_job_up_gives_way(shim, what):
    """A job runs in the memory that it cannot do without: no visit log where it would
    take the outputs' memory, a log of earlier jobs freed for them, and no flat walk
    where its row offsets do not fit."""
    child(shim, what)


def test_a_visit_log_is_allocated_when_it_pays(shim):
    """Jobs of few visits allocate nothing after an engine's first one, until as many
    visits were counted directly as cost what a log's allocation does."""
    child(shim, "later_jobs")


def test_only_larger_results_pin_memory(shim):
    """Results of up to 256 KB pin no memory, larger ones in an engine's first such job
    only, and once more when 32 MB of results of 4 MB or more went through that ring."""
    child(shim, "rings")


@pytest.mark.parametrize("what", ["no_ring", "no_query_table"])
def test_jobs_without_more_pinned_memory(shim, what):
    """Large results and query tables whose pinned memory cannot be had."""
    child(shim, what)


@pytest.mark.parametrize("slots", [0, 99])
def test_block_slots_where_raw_columns_do_not_fit(shim, slots):
    """Slots for all partitions, in memory that holds their block images only."""
    child(shim, "blocks", slots)


def test_the_cache_takes_what_its_layout_says(shim):
    """The bytes of lt_partition_slot_layout, or with block images and slots for all
    partitions the raw columns, within the raw slots asked for."""
    child(shim, "layout")


@pytest.mark.parametrize("form", ["flat", "queues", "learned"])
def test_after_failed_loads(shim, form):
    """Jobs that end at a partition copy's error, more of them than the cache has slots:
    the slots are there for the next job."""
    child(shim, "loads", form)


# ---- the child process ------------------------------------------------------------

FORMS = {"flat": dict(span="resident", resident_batch=16, zerocopy_threshold=0),
         "queues": dict(num_device_partitions=3, span="resident"),
         "spill": dict(num_device_partitions=3, num_device_walkers=9000),
         "batch": dict(num_device_partitions=3),
         "device": dict(num_device_partitions=3, device_schedule=1),
         "learned": dict(num_device_partitions=4, span="resident", policy="learned", prefetch_plain=1,
                         prefetch_depth=2, zerocopy_threshold=0)}


class Child:
    def __init__(self, path):
        self.lib = ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)
        self.lib.hipfail_held.restype = ctypes.c_size_t
        self.lib.hipfail_failed.restype = self.lib.hipfail_calls.restype = ctypes.c_long
        sys.path.insert(0, ROOT)
        import numpy as np

        import lighttraffic_amd as lt
        from oracle import ffi as oracle
        self.np, self.lt, self.oracle = np, lt, oracle
        self.graph = lt.Graph.rmat(13, 8)
        self.rp, self.col = self.graph.rowptr(), self.graph.col()
        self.part = lt.Partition.build(self.graph, 32 << 10)
        assert self.part.count > 8

    def arm(self, kind, skip=0, times=1, least=0, most=1 << 62):
        self.lib.hipfail_arm(ctypes.c_int(kind), ctypes.c_long(skip), ctypes.c_long(times), ctypes.c_size_t(least),
                             ctypes.c_size_t(most))

    def disarm(self, kind):
        n = self.lib.hipfail_failed(kind)
        self.arm(kind, times=0)
        return n

    def held(self):
        return self.lib.hipfail_held()

    def limit(self, n):
        self.lib.hipfail_limit(ctypes.c_size_t(n))

    def engine(self, **kw):
        return self.lt.Engine(self.graph, self.part, **kw)

    def jobs(self, eng, w, batch=False):
        """Jobs of every kind with w walkers; wrong values raise AssertionError."""
        np, o, rp, col = self.np, self.oracle, self.rp, self.col
        if batch:
            src, cnt = np.arange(7, dtype=np.uint32), np.full(7, w // 7 + 1, np.uint64)
            assert np.array_equal(eng.ppr_batch(src, cnt), o.ppr_batch(rp, col, src, cnt, threads=8)[0])
            return
        counts, ends = eng.pagerank(w, 4, endpoints=True)
        rc, re, _ = o.pagerank(rp, col, w, 4, endpoints=True, threads=8)
        assert np.array_equal(counts, rc) and np.array_equal(ends, re)
        ends, moves = eng.genericwalk(w, 3, moves=True)
        re, rm, _ = o.genericwalk(rp, col, w, 3, threads=8)
        assert np.array_equal(ends, re) and np.array_equal(moves, rm)
        assert np.array_equal(eng.genericwalk_paths(w, 3), o.genericwalk_paths(rp, col, w, 3))

    def after(self, form):
        small, large, n = 5000, 60000, 0
        while True:
            eng = self.engine(**FORMS[form])
            self.jobs(eng, small, form == "batch")
            self.arm(MALLOC, skip=n)
            try:
                self.jobs(eng, large, form == "batch")
            except self.lt.LTError as e:
                assert e.status == 4, e  # LT_E_NOMEM
            failed = self.disarm(MALLOC)
            print(form, "allocation", n, "failed" if failed else "was not made", flush=True)
            for w in (small + 1000, small, large):
                self.jobs(eng, w, form == "batch")
            eng.close()
            if not failed:
                assert n > 2
                return
            n += 1

    def pagerank(self, eng, w, l):
        counts, ends = eng.pagerank(w, l, endpoints=True)
        rc, re, _ = self.oracle.pagerank(self.rp, self.col, w, l, endpoints=True, threads=16)
        assert self.np.array_equal(counts, rc) and self.np.array_equal(ends, re)
        return eng.stats()

    W, L = 1200000, 30  # 36 M visits

    def logged(self):
        """A flat engine with its graph cached, and the bytes that it holds once it
        has also counted W * L visits through a log."""
        engines = [self.engine(**FORMS["flat"]) for _ in range(2)]
        for eng in engines:
            self.pagerank(eng, self.part.count * 4096, 3)
            before = self.held()
        assert self.pagerank(engines[1], self.W, self.L)["iterations"] == 1
        assert self.held() - before > 1 << 28  # with a log
        return engines, self.held() - before

    def log(self):
        (eng, other), most = self.logged()
        other.close()
        base = self.held()
        for less in (1, 4 * self.W, most // 2):
            self.limit(base + most - less)
            self.pagerank(eng, self.W, self.L)
        self.limit(1 << 62)
        self.pagerank(eng, self.W, self.L)
        assert self.held() - base == most

    def kept_log(self):
        (_, eng), _ = self.logged()
        held = self.held()
        self.limit(held)
        assert self.np.array_equal(eng.genericwalk_paths(60000, 9),
                                   self.oracle.genericwalk_paths(self.rp, self.col, 60000, 9))
        assert self.held() < held
        self.pagerank(eng, self.W, self.L)

    def offsets(self):
        eng = self.engine(**FORMS["flat"])
        n = 4 * (self.graph.num_node + 1)
        self.arm(MALLOC, times=1 << 40, least=n, most=n)
        w = self.part.count * 4096
        for _ in range(2):
            assert self.pagerank(eng, w, 4)["iterations"] > 1
        assert self.disarm(MALLOC) > 0
        assert self.pagerank(eng, w, 4)["iterations"] == 1

    def later_jobs(self):
        eng = self.engine(**FORMS["flat"])
        w, l = 100000, 10  # 1 M visits
        self.pagerank(eng, w, l)
        held = self.held()
        paid = 0
        for job in range(2, 41):
            assert self.pagerank(eng, w, l)["iterations"] == 1
            if self.held() != held:
                assert not paid and job * w * l >= 1 << 25 > (job - 1) * w * l
                held, paid = self.held(), job
        assert paid
        eng = self.engine(**FORMS["flat"])  # one job of that many
        self.pagerank(eng, self.part.count * 4096, 2)
        held = self.held()
        self.pagerank(eng, self.W, self.L)
        assert self.held() - held > 1 << 28
        held = self.held()
        self.pagerank(eng, w, l)  # small ones use it
        assert self.held() == held

    def rings(self):
        eng = self.engine(**FORMS["flat"])
        for _ in range(2):
            eng.genericwalk(30000, 9)

        def pins(w):
            self.arm(HOST_MALLOC, times=0)
            ends, moves = eng.genericwalk(w, 3, moves=True)
            re, rm, _ = self.oracle.genericwalk(self.rp, self.col, w, 3, threads=16)
            assert self.np.array_equal(ends, re) and self.np.array_equal(moves, rm)
            return self.lib.hipfail_calls(HOST_MALLOC)

        assert [pins(w) for w in (32768, 32769, 70000, 900000, 1 << 20, 1 << 20, 70000)] == [0, 1, 0, 0, 0, 0, 0]
        assert sum(pins(1500000) for _ in range(12)) == 1  # when the first ring is ready and 32 MB went through
        assert [pins(w) for w in (70000, 1500000, 1 << 21)] == [0, 0, 0]

    def no_ring(self):
        for kw in (FORMS["flat"], FORMS["queues"]):
            eng = self.engine(**kw)
            self.arm(HOST_MALLOC, times=1 << 40)
            for w in (70000, 1200000):
                ends, moves = eng.genericwalk(w, 3, moves=True)
                re, rm, _ = self.oracle.genericwalk(self.rp, self.col, w, 3, threads=16)
                assert self.np.array_equal(ends, re) and self.np.array_equal(moves, rm)
            assert self.disarm(HOST_MALLOC) > 0
            assert self.np.array_equal(eng.genericwalk(3000000, 3)[0][:w], re)

    def no_query_table(self):
        eng = self.engine(**FORMS["flat"])
        self.arm(HOST_MALLOC, times=1 << 40)
        self.jobs(eng, 5000, batch=True)
        assert self.disarm(HOST_MALLOC) > 0
        self.jobs(eng, 5000, batch=True)

    def blocks(self, slots):
        kw = dict(FORMS["flat"], pack_partitions=2, num_device_partitions=int(slots))
        assert self.part.count <= 99
        size, n = self.part.slot_layout(self.graph, 2, int(slots))
        raw = 8 * (self.graph.num_node + 1) + 4 * self.graph.num_edge
        assert n == self.part.count and n * size < raw
        self.arm(MALLOC, times=1 << 40, least=raw, most=raw + 255)
        eng = self.engine(**kw)
        assert self.disarm(MALLOC) == 1
        self.jobs(eng, 60000)
        st = eng.stats()
        assert st["cache_slots"] == n and st["iterations"] > 1  # by queues
        self.jobs(self.engine(**kw), 60000)

    def layout(self):
        P, raw = self.part.count, 8 * (self.graph.num_node + 1) + 4 * self.graph.num_edge

        def made(pack, slots, least, most):
            """Allocations of that size by an engine's creation."""
            self.arm(MALLOC, times=0, least=least, most=most)
            self.engine(pack_partitions=pack, num_device_partitions=slots).close()
            return self.lib.hipfail_calls(MALLOC)

        for pack, slots in ((0, 3), (1, 3), (2, 3), (2, P // 2)):
            size, n = self.part.slot_layout(self.graph, pack, slots)
            assert made(pack, slots, n * size, n * size) == 1, (pack, slots)
        for slots in (0, P, 99):
            size, n = self.part.slot_layout(self.graph, 2, slots)
            raw_size, raw_n = self.part.slot_layout(self.graph, 0, slots)
            assert n == raw_n == P and n * size < raw <= raw + 255 <= raw_n * raw_size
            assert made(2, slots, raw, raw + 255) == 1 and made(2, slots, raw + 256, 1 << 62) == 0

    def loads(self, form):
        eng = self.engine(pack_partitions=1, **FORMS[form])
        w = self.part.count * 4096
        for n in range(2 * self.part.count + 3):
            self.arm(MEMCPY_ASYNC, skip=n)
            try:
                self.pagerank(eng, w, 3)
            except self.lt.LTError as e:
                assert e.status == 5, e  # LT_E_HIP
            self.disarm(MEMCPY_ASYNC)
        for _ in range(2):
            self.jobs(eng, w)


if __name__ == "__main__":
    c = Child(sys.argv[1])
    getattr(c, sys.argv[2])(*sys.argv[3:])
    print("done", flush=True)
