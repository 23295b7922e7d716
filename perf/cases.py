"""Performance cases of the random-walk engine: the jobs its users run, called
through the package's public entry points on seeded graphs.

A case is a plain dict.  `kind` says which entry point it calls:

  pagerank / genericwalk / paths / ppr / ppr_batch
      one walk job on an engine that the program keeps (graph, partition table
      and engine are made once, jobs follow): Engine.pagerank and so on.
      scale, ef            R-MAT graph (2^scale ids, ef * 2^scale sampled edges)
      split, part_kb       "equal": Partition.build at part_kb KiB;
                           "blocks": Partition.build_blocks with part_kb KiB slots
      cache                share of the graph's partitions the HBM cache holds
                           (0: all of them)
      walks                walkers per vertex (for ppr_batch: queries)
      length               steps per walker (fixed-length kinds)
      the engine options of the same names, when given
  scorer_grad / scorer_infer
      the learned scheduler's network on `decisions` decisions over
      `partitions` partitions: Scorer.loss_grad, Scorer.infer

Sizes are this repository's benchmark and test configurations (R-MAT s10 ef8,
s16 ef16, s22 ef16, and the s25 ef44 and s26 ef27 workloads scaled down with
their partition size so that the partition counts and the cached share stay
what they are there).
"""
import math

import numpy as np
import torch

import lighttraffic_amd as lt

MB = 1024  # KiB

# Engine options a case may carry.
OPTIONS = ("span", "policy", "zc_batch", "resident_batch", "pack_partitions", "prefetch_plain", "prefetch_depth",
           "walkers_per_thread", "rowptr_resident", "device_schedule", "slice_chunks")


def listed():
    return [
        # The smallest job: a graph of a few hundred vertices, cached; what a
        # call costs beyond its walk.
        dict(name="pagerank_s10", kind="pagerank", scale=10, ef=8, split="equal", part_kb=32 * MB, cache=0.0,
             zc_threshold=0, walks=2.0, length=10),
        # One cached 32 MB partition (the benchmark's c1).
        dict(name="pagerank_s16", kind="pagerank", scale=16, ef=16, split="equal", part_kb=32 * MB, cache=0.0,
             zc_threshold=0, walks=2.0, length=10),
        # A graph that fits the HBM cache whole, walked through every partition.
        dict(name="pagerank_s22", kind="pagerank", scale=22, ef=16, split="equal", part_kb=32 * MB, cache=0.0,
             walks=2.0, length=10, span="resident", resident_batch=16),
        # The same for fixed-length walks with their endpoints (the benchmark's c2).
        dict(name="generic_s22", kind="genericwalk", scale=22, ef=16, split="equal", part_kb=32 * MB, cache=0.0,
             walks=2.0, length=10, span="resident", resident_batch=16, walkers_per_thread=2),
        # Whole paths, as a corpus for embedding training; an odd walker count.
        dict(name="paths_s17", kind="paths", scale=17, ef=16, split="equal", part_kb=4 * MB, cache=0.0,
             zc_threshold=0, walks=1.0001, length=40),
        # Personalised pagerank of one vertex with a third of the graph cached
        # (the benchmark's c3: balanced split, prefetch, zero-copied leftovers).
        dict(name="ppr_s20_third", kind="ppr", scale=20, ef=44, split="blocks", part_kb=1 * MB, cache=0.6,
             walks=2.0, span="resident", policy="learned", prefetch_plain=1, zc_batch=16, resident_batch=16,
             pack_partitions=2, walkers_per_thread=1, rowptr_resident=1, zc_div=128),
        # Batched personalised pagerank, every block slot cached (the benchmark's
        # c4 as its autotuner sets it).
        dict(name="pprbatch_s20", kind="ppr_batch", scale=20, ef=44, split="blocks", part_kb=2 * MB, cache=0.0,
             walks=128, lo=1000, hi=200000, span="resident", zc_batch=16, resident_batch=16, pack_partitions=2,
             walkers_per_thread=1, slice_chunks=8192),
        # A graph larger than the cache with everything tuned (the benchmark's
        # c5 loop: balanced split, block slots, prefetch of the largest queues).
        dict(name="pagerank_s23_capped", kind="pagerank", scale=23, ef=27, split="blocks", part_kb=4 * MB,
             cache=0.87, walks=2.0, length=10, span="resident", policy="learned", prefetch_plain=1,
             prefetch_depth=2, zc_batch=16, resident_batch=16, pack_partitions=2, walkers_per_thread=1, zc_div=128),
        # The same kind of graph under the reference's own rules and defaults:
        # raw copies, one partition at a time.
        dict(name="pagerank_s20_plain", kind="pagerank", scale=20, ef=27, split="equal", part_kb=2 * MB, cache=0.6,
             walks=2.0, length=10),
        # Scheduling on the GPU: decisions, copies and walks in one captured graph.
        dict(name="generic_s18_device", kind="genericwalk", scale=18, ef=16, split="equal", part_kb=1 * MB,
             cache=0.6, walks=2.0, length=10, device_schedule=1),
        # One training step of the learned scheduler's network (the benchmark
        # trains it on batches of 32 decisions over c5's partitions).
        dict(name="scorer_grad_32x291", kind="scorer_grad", decisions=32, partitions=291),
        # One decision scored.
        dict(name="scorer_infer_291", kind="scorer_infer", decisions=1, partitions=291),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["pagerank", "pagerank", "pagerank", "genericwalk", "genericwalk", "paths", "ppr", "ppr_batch",
                       "scorer_grad", "scorer_infer"])
    if kind == "scorer_grad":
        return dict(kind=kind, decisions=int(_log_uniform(rng, 1, 33)), partitions=int(_log_uniform(rng, 5, 450)))
    if kind == "scorer_infer":
        return dict(kind=kind, decisions=1, partitions=int(_log_uniform(rng, 5, 20000)))
    # the cache: everything resident (with or without walking through all of
    # it), the reference's rules, or the tuned loop
    mode = rng.choice(["resident", "resident", "fits", "plain", "tuned"])
    # ids up to 2^21, less where a pass returns whole paths or waits for the host link
    scale = rng.randint(10, 17 if kind == "paths" else 18 if mode in ("plain", "tuned") else 21)
    ef = rng.randint(4, 27) if scale > 20 else rng.randint(4, 44)
    c = dict(kind=kind, scale=scale, ef=ef, walks=round(rng.uniform(0.5, 2.5), 4))
    kib = 2 * ef * 2.0 ** scale * 4 / 1024  # about the columns' size
    if mode in ("plain", "tuned"):  # 12 to 250 partitions, 0.5 to 0.9 of them cached
        c["part_kb"] = max(32, int(kib / _log_uniform(rng, 12, 250)))
        c["cache"] = round(rng.uniform(0.5, 0.9), 3)
    else:
        c["part_kb"] = max(64, int(kib / _log_uniform(rng, 1, 60)))
        c["cache"] = 0.0
    c["split"] = "equal"
    if mode == "resident":
        c.update(span="resident", resident_batch=16, walkers_per_thread=rng.choice([0, 1, 2, 4]))
        if rng.random() < 0.7:  # else the default threshold: small queues are read over PCIe
            c["zc_threshold"] = 0
    elif mode == "tuned":
        c.update(split="blocks", span="resident", policy="learned", prefetch_plain=1, zc_batch=16, resident_batch=16,
                 pack_partitions=2, walkers_per_thread=1, zc_div=128, rowptr_resident=rng.choice([0, 1]))
    elif mode == "fits":
        c.update(zc_threshold=rng.choice([0, 4096]), pack_partitions=rng.choice([0, 0, 2]))
    else:
        c.update(pack_partitions=rng.choice([0, 0, 1, 2]))
    if kind in ("pagerank", "genericwalk"):
        c["length"] = rng.randint(3, 20) if scale <= 20 else rng.randint(3, 10)
    elif kind == "paths":
        c["length"] = rng.randint(5, 40)
    elif kind == "ppr_batch":
        c.update(walks=rng.randint(8, 128), lo=1000, hi=int(_log_uniform(rng, 2000, 100000)))
    return c


# ---- walk jobs ------------------------------------------------------------------

def _walk_state(case, seed):
    # the generator's graph of this scale and edge factor; the seed gives the
    # walks (and the queries' sources), so that every pass returns as many values
    graph = lt.Graph.rmat(case["scale"], case["ef"])
    size = int(case["part_kb"]) * 1024
    # the largest row bounds the partition size from below
    row = int(np.diff(graph.rowptr()).max()) * 4 + 64
    size = max(size, row)
    part = lt.Partition.build_blocks(graph, size) if case["split"] == "blocks" else lt.Partition.build(graph, size)
    opts = {k: case[k] for k in OPTIONS if k in case}
    if case["cache"]:
        slots = max(2, int(part.count * case["cache"]))
        if case["split"] == "blocks":  # the cache is given in raw slots; it holds `slots` block slots
            slots = max(2, int(slots * size / part.bytes))
        opts["num_device_partitions"] = slots
    if "zc_threshold" in case:
        opts["zerocopy_threshold"] = case["zc_threshold"]
    elif "zc_div" in case:
        opts["zerocopy_threshold"] = size // case["zc_div"]
    engine = lt.Engine(graph, part, seed=0x4C540000 + int(seed), **opts)
    state = dict(kind=case["kind"], engine=engine, length=case.get("length", 0),
                 w=max(1, int(case["walks"] * graph.num_node)))
    if case["kind"] == "ppr":
        state["source"] = 0
    if case["kind"] == "ppr_batch":
        nq = int(case["walks"])
        sources = graph.ppr_queries(nq, case["lo"], case["hi"], seed=0x51520000 + int(seed))[0]
        state["queries"] = sources, graph.ppr_queries(nq, case["lo"], case["hi"])[1]
    return state


# ---- the scheduler's network -------------------------------------------------------

HIDDEN, FEATURES, OUTPUTS, RECENT = 256, 16, 2, 8
SIZES = ((FEATURES, HIDDEN), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,), (HIDDEN, OUTPUTS), (OUTPUTS,))


def _parameters(rng):
    """FP32 weights and small biases, as an initialised and partly trained network has them."""
    out = []
    for shape in SIZES:
        scale = math.sqrt(2.0 / shape[0]) if len(shape) == 2 else 0.05
        out.append((rng.standard_normal(int(np.prod(shape))) * scale).astype(np.float32))
    return np.concatenate(out)


def _table(partitions):
    """A partition table of that many partitions over a ring whose rows hold one or two edges."""
    per = 6
    n = partitions * per
    degree = 1 + (np.arange(n) % 3 == 0)
    rowptr = np.concatenate([[0], np.cumsum(degree)]).astype(np.uint64)
    col = ((np.arange(int(rowptr[-1])) * 7) % n).astype(np.uint32)
    graph = lt.Graph.from_csr(rowptr, col)
    part = lt.Partition.build(graph, (per + 1) * 8 + 8 * 4)
    return graph, part


def _decisions(case, seed):
    """Queue lengths, residency, ages and labels of decisions: most queues are
    empty, the others spread over three orders of magnitude."""
    rng = np.random.default_rng([int(seed), 77])
    P = int(case["partitions"])
    params = _parameters(rng)
    samples = []
    for i in range(int(case["decisions"])):
        resident = (rng.random(P) < 0.8).astype(np.uint8)
        counts = np.exp(rng.uniform(0, 12, P)).astype(np.uint32)
        counts[(rng.random(P) < 0.8) & (resident != 0)] = 0
        recent = rng.integers(-1, P, RECENT).astype(np.int32)
        samples.append(dict(counts=counts, resident=resident, age=rng.integers(0, 3 * P, P).astype(np.uint32),
                            recent=recent, cur=int(rng.integers(0, P)), w_total=float(counts.sum()) * 1.5 + 1.0,
                            next=int(np.argmax(counts)) if i % 4 != 3 else -1,
                            keep=rng.random(P).astype(np.float32), wa=1.0 if i % 4 != 3 else 0.0, wb=1.0))
    return params, samples


def prepare(case, seed):
    if case["kind"] not in ("scorer_grad", "scorer_infer"):
        return _walk_state(case, seed)
    graph, part = _table(int(case["partitions"]))
    params, samples = _decisions(case, seed)
    scorer = lt.Scorer(part, seed=1)
    scorer.set_params(params)
    return dict(kind=case["kind"], graph=graph, part=part, scorer=scorer, samples=samples)


def run(state):
    kind = state["kind"]
    if kind == "scorer_grad":
        return state["scorer"].loss_grad(state["samples"])
    if kind == "scorer_infer":
        s = state["samples"][0]
        return state["scorer"].infer(s["counts"], s["resident"], s["age"], s["recent"], s["cur"], s["w_total"])
    engine = state["engine"]
    if kind == "pagerank":
        return engine.pagerank(state["w"], state["length"])
    if kind == "genericwalk":
        return engine.genericwalk(state["w"], state["length"], endpoints=True)[0]
    if kind == "paths":
        return engine.genericwalk_paths(state["w"], state["length"])
    if kind == "ppr":
        return engine.ppr(state["w"], source=state["source"], prob=0.15, endpoints=True)
    sources, counts = state["queries"]
    return engine.ppr_batch(sources, counts, prob=0.15, endpoints=True)


def work(case):
    """Bytes a pass cannot do without: of the graph what its moves read, 20
    bytes a move and each byte once at most; the results once.  Vertex and
    edge counts are the generator's usual shares of 2^scale and ef * 2^scale."""
    if case["kind"] == "scorer_grad":
        rows = case["decisions"] * case["partitions"]
        macs = FEATURES * HIDDEN + HIDDEN * HIDDEN + HIDDEN * OUTPUTS
        params = sum(int(np.prod(s)) for s in SIZES)
        # forward, weight gradients, and the input gradients of the upper two layers
        flops = 2 * rows * (2 * macs + HIDDEN * HIDDEN + HIDDEN * OUTPUTS)
        return dict(bytes=rows * 13 + params * 8, flops=flops)
    if case["kind"] == "scorer_infer":
        rows = case["partitions"]
        macs = FEATURES * HIDDEN + HIDDEN * HIDDEN + HIDDEN * OUTPUTS
        return dict(bytes=rows * 25 + sum(int(np.prod(s)) for s in SIZES) * 2, flops=2 * rows * macs)
    V = 0.6 * 2.0 ** case["scale"]
    E = 1.8 * case["ef"] * 2.0 ** case["scale"]
    graph = 8 * V + 4 * E
    kind = case["kind"]
    if kind == "ppr_batch":
        walkers = case["walks"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
    else:
        walkers = case["walks"] * V
    if kind == "pagerank":
        moves, result = walkers * (case["length"] - 1) * 0.85, 4 * V
    elif kind == "genericwalk":
        moves, result = walkers * case["length"], 4 * walkers
    elif kind == "paths":
        moves, result = walkers * case["length"], 4 * walkers * (case["length"] + 1)
    else:  # 2 + a geometric number of draws
        moves = walkers * (1 + 0.85 / 0.15)
        result = 4 * walkers + (4 * V if kind == "ppr" else 0)
    return dict(bytes=min(20 * moves, graph) + result, flops=0)


# ---- 64-bit values of what the network computes ----------------------------------------

def _features(s, vertex_share, edge_share):
    c = torch.from_numpy(s["counts"].astype(np.float64))
    P = len(c)
    w = max(float(np.float32(s["w_total"])), 1.0)
    x = torch.zeros(P, FEATURES, dtype=torch.float64)
    x[:, 0] = torch.log1p(c) / math.log1p(w)
    x[:, 1] = c / max(float(c.max()), 1.0)
    x[:, 2] = torch.log1p(c / max(float(c.sum()) / P, 1.0))
    x[:, 3] = torch.from_numpy((s["resident"] != 0).astype(np.float64))
    x[s["cur"], 4] = 1.0
    for k in range(RECENT - 1):
        if s["recent"][k] >= 0:
            x[s["recent"][k], 5 + k] = 1.0
    age = torch.from_numpy(s["age"].astype(np.float64))
    x[:, 12] = age / (age + P)
    x[:, 13] = vertex_share
    x[:, 14] = edge_share
    x[:, 15] = float(c.sum()) / w
    return x


def _rounded(params):
    """The network's products use the weights rounded to bfloat16."""
    out, off = [], 0
    for shape in SIZES:
        n = int(np.prod(shape))
        t = torch.from_numpy(params[off:off + n]).to(torch.bfloat16).to(torch.float64).reshape(shape)
        out.append(t.requires_grad_())
        off += n
    return out


def exact(case, seed):
    """Walk jobs return whole numbers and have no such value; the network's
    outputs are computed again in 64 bits."""
    if case["kind"] not in ("scorer_grad", "scorer_infer"):
        return None
    P = int(case["partitions"])
    params, samples = _decisions(case, seed)
    ring = 1 + (np.arange(P * 6) % 3 == 0)
    # every partition holds the same six vertices and eight edges
    share = ring.reshape(P, 6).sum(1) / ring.sum() * P
    vertex_share, edge_share = torch.ones(P, dtype=torch.float64), torch.from_numpy(share)
    w1, b1, w2, b2, w3, b3 = weights = _rounded(params)
    B = len(samples)
    first = torch.zeros((), dtype=torch.float64)
    second = torch.zeros((), dtype=torch.float64)
    for s in samples:
        x = _features(s, vertex_share, edge_share)
        y = torch.relu(torch.relu(x @ w1 + b1) @ w2 + b2) @ w3 + b3
        if case["kind"] == "scorer_infer":
            return y.detach().numpy()
        if s["next"] >= 0 and s["wa"] > 0:
            cand = torch.from_numpy(s["counts"] > 0)
            cand[s["next"]] = True
            first = first + s["wa"] * (torch.logsumexp(y[cand, 0], 0) - y[s["next"], 0]) / B
        keep = torch.from_numpy(s["keep"].astype(np.float64))
        second = second + s["wb"] * ((y[:, 1] - keep) ** 2).sum() / B / P
    (first + second).backward()
    grad = np.concatenate([t.grad.numpy().ravel() for t in weights])
    return np.array([first.item(), second.item()]), grad
