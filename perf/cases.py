"""The work that users of this framework have it do, as measurable cases.

A program builds a kNN graph (GNN-Descent), prunes it into an index (NSG, Vamana, NSSG, CAGRA
or DPG) and searches the index; the clustered large-index pipeline builds and prunes many
uneven clusters packed into one handle.  Each case is one such call, or the build-and-prune
pair, on a handle that already holds its vectors (and its graph or index where the call starts
from one).

Vectors come from the framework's own seeded generator: "int" are integer-valued clipped
mixtures in [0, 255] (bytes-like descriptors), "unit" L2-normalised mixtures (embeddings),
"abs" non-negative wide vectors scaled to [0, 1].  `prepare(case, seed)` derives both the
vectors and the algorithm's random streams from the seed.
"""
import math

import numpy as np
import torch

from tagore_amd import State

GEN = {"int": 0, "unit": 1, "abs": 2}
# index -> (kind, forward rule, reverse rule, threshold)
INDEX = {
    "nsg": ("path", "dist", "dist", 1.0),
    "vamana": ("path", "dist", "dist", 1.2),
    "nssg": ("2-hop", "angle", "angle", 0.5),
    "cagra": ("cagra", "dist", "rank", 0.0),
    "dpg": ("dpg", "dist", "rank", 0.0),
}


def listed():
    return [
        # one query against a 100k index: a serving call, where the call's own cost counts
        dict(name="search_one", op="search", data="int", n=100_000, d=128, comps=100, k=48,
             index="nsg", fd=32, m=64, nq=1, pool=64, topk=10),
        # a batch of held-out queries against the million-vector index
        dict(name="search_batch", op="search", data="int", n=1_000_000, d=128, comps=1024, k=96,
             index="nsg", fd=32, m=64, nq=10_000, pool=64, topk=10),
        # the 10k x 128 plain FP32 configuration in full: build from random lists, then NSG
        dict(name="small_full", op="both", data="int", n=10_000, d=128, comps=64, k=32, iters=10,
             precision="fp32", init="random", index="nsg", fd=32, m=64),
        # the million-vector build: learned lists, BF16 screen, 2 iterations
        dict(name="knn_learned_1m", op="knn", data="int", n=1_000_000, d=128, comps=1024, k=96,
             iters=2, precision="bf16", init="learned", sample=25_000, epochs=1),
        # NSG over that graph
        dict(name="nsg_1m", op="prune", data="int", n=1_000_000, d=128, comps=1024, k=96,
             index="nsg", fd=32, m=64),
        # Vamana (alpha 1.2) keeps long candidate lists alive through the filter
        dict(name="vamana_int", op="prune", data="int", n=400_000, d=128, comps=400, k=96,
             index="vamana", fd=32, m=64),
        # the one-hop rank rule, no distances
        dict(name="cagra_int", op="prune", data="int", n=500_000, d=128, comps=512, k=96,
             index="cagra", fd=32, m=64),
        # embeddings: learned lists (five epochs), 4 iterations, real-valued rows
        dict(name="knn_unit", op="knn", data="unit", n=500_000, d=96, comps=256, k=64, iters=4,
             precision="bf16", init="learned", sample=50_000, epochs=5),
        # two-hop / angle over embeddings, an odd number of rows
        dict(name="nssg_unit", op="prune", data="unit", n=299_993, d=96, comps=153, k=50,
             index="nssg", fd=32, m=64),
        # uneven clusters in one handle: 8+8 iterations from random lists, Vamana each
        dict(name="clusters_full", op="both", data="unit", n=160_003, d=96, comps=64, k=64,
             iters=16, precision="bf16", init="random", index="vamana", fd=32, m=64,
             segments=12),
        # wide rows: 960 dimensions
        dict(name="knn_wide", op="knn", data="abs", n=100_000, d=960, comps=64, k=64, iters=4,
             precision="bf16", init="learned", sample=25_000, epochs=2),
        # occlusion counts on wide rows
        dict(name="dpg_wide", op="prune", data="abs", n=100_000, d=960, comps=64, k=64,
             index="dpg", fd=32, m=64, rows="bf16"),
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["search", "knn", "prune", "both"])
    data = rng.choice(["int", "int", "unit", "unit", "abs"])
    d = {"int": lambda: 4 * rng.randint(16, 40), "unit": lambda: 8 * rng.randint(8, 20),
         "abs": lambda: 32 * rng.randint(8, 30)}[data]()
    most = {"int": 600_000, "unit": 250_000, "abs": 60_000}[data]
    n = _log(rng, 5_000, most)
    k = rng.randint(24, 96 if data == "int" else 64)
    c = dict(op=op, data=data, n=n, d=d, comps=max(8, n // 1000), k=k)
    if op in ("knn", "both"):
        learned = d % 32 == 0 and rng.random() < 0.6 and op == "knn"
        c["precision"] = rng.choice(["fp32", "bf16", "exact"] if d % 8 == 0 else ["fp32", "exact"])
        c["init"] = "learned" if learned else "random"
        c["iters"] = 2 * rng.randint(1, 3) if learned else 2 * rng.randint(2, 4)
        if learned:
            c.update(sample=min(n, 25_000), epochs=rng.randint(1, 3))
        else:
            c["n"] = min(n, most // 3 + n % 4096)
    if op != "knn":
        c["index"] = rng.choice(["nsg", "vamana", "nssg", "cagra", "dpg"]
                                if op != "search" else ["nsg", "vamana", "nssg"])
        c["fd"] = rng.randint(16, min(k, 48))
        c["m"] = rng.randint(32, 80)
        if c["index"] == "dpg" and d % 8 == 0 and k <= 64:
            c["rows"] = "bf16"
    if op == "both" and rng.random() < 0.4:
        c["segments"] = rng.randint(2, 9)
    if op == "search":
        c.update(nq=_log(rng, 1, 10_000), pool=rng.randint(12, 128), topk=10)
    return c


def _segment_starts(n, count, k):
    """Starts of `count` log-normal segments over n rows (no segment below k + 1 rows)."""
    w = np.random.default_rng(n).lognormal(0.0, 0.945, count)
    w = np.clip(w / np.median(w), 0.125, 5.0)
    least = min(n // count, 4 * (k + 1))
    size = least + ((n - least * count) * w / w.sum()).astype(np.int64)
    size[0] += n - size.sum()
    return np.concatenate([[0], np.cumsum(size)]).astype(np.uint32)


def _build(st, case, seed):
    st.knn_build(case["k"], case["iters"], seed, case["precision"], init=case["init"],
                 sample=case.get("sample", 0), epochs=case.get("epochs", 0))


def _prune(st, case):
    kind, fwd, rev, th = INDEX[case["index"]]
    st.prune(kind, fwd, rev, case["fd"], case["m"], th, case.get("rows", "fp32"))


def prepare(case, seed):
    n, d, nq = case["n"], case["d"], case.get("nq", 0)
    st = State(n, d)
    st.gen_data(GEN[case["data"]], case["comps"], seed, 20.0)
    queries = None
    if case["op"] == "search":
        # held-out queries: the generator's next vectors
        with State(n + nq, d) as g:
            g.gen_data(GEN[case["data"]], case["comps"], seed, 20.0)
            queries = g.get_data(n, nq)
    if case.get("segments"):
        st.set_segments(_segment_starts(n, case["segments"], case["k"]))
    if case["op"] in ("search", "prune"):
        # the graph (and index) that the call starts from
        learned = d % 32 == 0
        st.knn_build(case["k"], 2 if learned else 8, seed,
                     "bf16" if d % 8 == 0 else "fp32", init="learned" if learned else "random",
                     sample=min(n, 25_000) if learned else 0, epochs=1 if learned else 0)
        if case["op"] == "search":
            _prune(st, case)
    return dict(case=case, seed=seed, st=st, queries=queries)


class _DeviceArray:
    """A handle's device buffer for torch.as_tensor; keeps the handle alive."""

    def __init__(self, st, idx, shape, dtype):
        ptr, _ = st.buffer(idx)
        self.owner = st
        self.__cuda_array_interface__ = dict(shape=shape, typestr=dtype, data=(ptr, False),
                                             version=2)


def _graph(st, case):
    """The kNN graph where it is: device ids and distances, as a later step reads them."""
    shape = (case["n"], case["k"])
    return {"ids": torch.as_tensor(_DeviceArray(st, 0, shape, "<i4"), device="cuda"),
            "dists": torch.as_tensor(_DeviceArray(st, 3, shape, "<f4"), device="cuda")}


def _pruned(st):
    deg, ids, ep = st.get_pruned()
    return {"deg": deg.view(np.int32), "adj": ids.view(np.int32), "ep": ep}


def run(state):
    case, st = state["case"], state["st"]
    if case["op"] == "search":
        ids, dists, stats = st.search(state["queries"], k=case["topk"], L=case["pool"],
                                      seed=state["seed"])
        return {"ids": ids.view(np.int32), "dists": dists, "evals": stats["evals"]}
    out = {}
    if case["op"] in ("knn", "both"):
        _build(st, case, state["seed"])
        out.update(_graph(st, case))
    if case["op"] in ("prune", "both"):
        _prune(st, case)
        out.update(_pruned(st))
    return out


def work(case):
    """Each input once, each output once; distances as 3 operations per dimension."""
    n, d, k = case["n"], case["d"], case["k"]
    fd, m = case.get("fd", 0), case.get("m", 0)
    rows, graph, index = n * d * 4, n * k * 8, n * (fd + 1) * 4
    if case["op"] == "search":
        nq, pool = case["nq"], case["pool"]
        evals = nq * pool * (1 + fd // 4)
        read = min(rows, evals * d * 4) + min(index, nq * pool * fd * 4)
        return {"bytes": read + nq * (d * 4 + case["topk"] * 8), "flops": 3 * d * evals}
    nbytes, evals = rows, 0
    if case["op"] in ("knn", "both"):
        # initial lists; sampled joins (32 + 32 samples); four leaders' lists per expansion
        half = case["iters"] // 2
        evals += n * (k + 2016 + (half - 1) * 4096 + half * 4 * min(64, k))
        nbytes += graph
    if case["op"] in ("prune", "both"):
        nbytes += graph + index
        if case["index"] in ("nsg", "vamana"):
            evals += n * (k + 10 * k // 2 + fd * (m + k) // 2)
        elif case["index"] == "nssg":
            evals += n * (480 + fd * (m + k) // 2)
        elif case["index"] == "dpg":
            evals += n * (k * (k - 1) // 2)
    return {"bytes": nbytes, "flops": 3 * d * evals}
