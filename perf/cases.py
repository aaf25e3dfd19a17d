"""The work a user of the partitioner has it do, as cases that can be timed.

A case names a call (`op`), a graph and the options of the call:

  partition    one whole multilevel partition of a resident graph (gp_partition)
  coarsen      the coarsening levels of a resident graph (gp_coarsen); the
               maps and the coarsest graph go back to the host, where the
               caller's own initial partitioner reads them
  uncoarsen    projection and refinement of a kept hierarchy from a coarsest
               partition (gp_uncoarsen)
  repartition  a resident graph takes a batch of new edges, its partition is
               refined from the one in hand, and the edges go again
               (gp_graph_apply_delta, gp_refine_partition)
  edge_cut     cut and part loads of labels in device memory (gp_edge_cut)
  serve        a batch of unequal host graphs through the request server
               (gp_server_submit, gp_server_wait)

Graphs: 4-neighbour grids, random geometric meshes of mean degree 8, R-MAT
graphs (a=0.57, b=c=0.19) and 3-D k-nearest-neighbour graphs with edge and
vertex weights: the generators of the tests and the benchmark.
"""
import functools
import importlib
import math
import random

import numpy as np
import torch

IMBALANCE = 1.03
R_MAT_KEPT = 0.92  # share of R-MAT's directed entries left after merging repeats (0.87 to 0.96)


def listed():
    return [
        # A tool partitioning a small mesh in a loop: launches and latency only.
        {"name": "partition_small", "op": "partition", "graph": "mesh", "n": 1501, "k": 4},
        # A regular 2-D discretisation on a quarter of a million cells.
        {"name": "partition_grid", "op": "partition", "graph": "grid", "rows": 511, "cols": 513, "k": 16},
        # An unstructured mesh split over a cluster; odd sizes throughout.
        {"name": "partition_mesh", "op": "partition", "graph": "mesh", "n": 777777, "k": 37},
        # A social-style graph of ordinary size: hub rows beside short ones.
        {"name": "partition_rmat", "op": "partition", "graph": "rmat", "scale": 18, "degree": 16, "k": 64},
        # The benchmark's graph, the largest one partitioned in one call.
        {"name": "partition_rmat_large", "op": "partition", "graph": "rmat", "scale": 22, "degree": 16, "k": 64},
        # A weighted particle graph at the largest number of parts.
        {"name": "partition_weighted", "op": "partition", "graph": "knn", "n": 300007, "k": 128},
        # Coarsening alone, for a caller with an initial partitioner of its own.
        {"name": "coarsen_rmat", "op": "coarsen", "graph": "rmat", "scale": 20, "degree": 12, "k": 32},
        # Refinement alone: many tries from one kept hierarchy.
        {"name": "uncoarsen_rmat", "op": "uncoarsen", "graph": "rmat", "scale": 19, "degree": 16, "k": 32},
        # A served mesh that changes a little and is repartitioned warm.
        {"name": "repartition_mesh", "op": "repartition", "graph": "mesh", "n": 262001, "k": 16, "changes": 10000},
        # The smallest call: judging a candidate partition of a small grid.
        {"name": "edge_cut_small", "op": "edge_cut", "graph": "grid", "rows": 64, "cols": 63, "k": 4},
        # The same on a large graph, bound by the memory it reads.
        {"name": "edge_cut_rmat", "op": "edge_cut", "graph": "rmat", "scale": 20, "degree": 16, "k": 64},
        # Unequal requests of the mixed workload, several in flight.
        {"name": "serve_mix", "op": "serve", "count": 18, "largest": 131072, "workers": 6},
    ]


def spread(rng, low, high):
    """A whole number between low and high, even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choice(["partition"] * 4 + ["coarsen", "uncoarsen", "repartition", "edge_cut", "serve"])
    if op == "serve":
        return {"op": op, "count": rng.randint(4, 24), "largest": spread(rng, 4096, 200000), "workers": rng.randint(2, 6)}
    kind = rng.choice(["grid", "mesh", "rmat", "knn"])
    case = {"op": op, "graph": kind}
    if kind == "grid":
        case["rows"], case["cols"] = spread(rng, 40, 1200), spread(rng, 40, 1200)
        n = case["rows"] * case["cols"]
    elif kind == "mesh":
        n = case["n"] = spread(rng, 1200, 1000000)
    elif kind == "rmat":
        case["scale"], case["degree"] = rng.randint(11, 20), rng.randint(6, 18)
        n = 1 << case["scale"]
    else:
        n = case["n"] = spread(rng, 2000, 400000)
    case["k"] = min(spread(rng, 2, 128), n // 64)
    if op == "repartition":
        case["changes"] = max(4, int(n * rng.uniform(0.005, 0.08)))
    return case


# ------------------------------------------------------------------ inputs
gp = importlib.import_module("acc-gp_amd")


@functools.lru_cache(maxsize=None)
def context():
    """One context for the program, as a caller keeps it."""
    return gp.Context(0)


@functools.lru_cache(maxsize=None)
def server(workers):
    return gp.Server(workers=workers)


def host_graph(case, seed):
    """(offsets, neighbours, edge weights, vertex weights) on the host.  A
    grid has no randomness of its own: there the seed is the partitioner's."""
    kind = case["graph"]
    if kind == "grid":
        return gp.generate_grid(case["rows"], case["cols"]) + (None, None)
    if kind == "mesh":
        return gp.generate_rgg2d(case["n"], math.sqrt(8.0 / (math.pi * case["n"])), seed=seed + 1) + (None, None)
    if kind == "rmat":
        return gp.generate_rmat(case["scale"], case["degree"], seed=seed + 1) + (None, None)
    return gp.generate_knn3d(case["n"], 10, seed=seed + 1)


class State:
    """What the caller holds; device objects go when it does."""

    def __init__(self, **kept):
        self.kept = kept

    def __getitem__(self, name):
        return self.kept[name]

    def __del__(self):
        for name in ("hierarchy", "graph"):  # the hierarchy borrows the graph
            if name in self.kept:
                self.kept[name].close()


def new_edges(off, nbr, count, rng):
    """`count` vertex pairs, none of them an edge yet and none twice (every
    generator gives ascending rows, so the edges' keys ascend)."""
    n = len(off) - 1
    there = np.repeat(np.arange(n, dtype=np.int64), np.diff(off)) * n + nbr
    u, v = rng.integers(0, n, 2 * count), rng.integers(0, n, 2 * count)
    key = np.unique((np.minimum(u, v) * n + np.maximum(u, v))[u != v])
    at = np.minimum(np.searchsorted(there, key), len(there) - 1)
    key = rng.permutation(key[there[at] != key])[:count]
    return (key // n).astype(np.int32), (key % n).astype(np.int32)


def serve_items(case, rng):
    """Grids, R-MAT graphs and meshes of up to `largest` vertices in turn.
    The case alone gives the sizes, the seed the graphs."""
    sizes = random.Random(case["count"] * 1000003 + case["largest"])
    items = []
    for i in range(case["count"]):
        n = spread(sizes, 1024, case["largest"])
        seed = int(rng.integers(1, 1 << 30))
        if i % 3 == 0:
            side = int(round(math.sqrt(n)))
            off, nbr = gp.generate_grid(side, side + sizes.randrange(8))
        elif i % 3 == 1:
            off, nbr = gp.generate_rmat(int(math.log2(n)), sizes.randrange(8, 17), seed=seed)
        else:
            off, nbr = gp.generate_rgg2d(n, math.sqrt(8.0 / (math.pi * n)), seed=seed)
        k = sizes.choice([4, 8, 16, 32, 64])
        while not feasible(len(off) - 1, k):
            k //= 2
        items.append(gp.BatchItem(off, nbr, k, IMBALANCE, seed=seed))
    return items


def feasible(n, k):
    """The integer capacity has to hold an even share."""
    return n >= 2 * k and math.floor(IMBALANCE * n / k) >= -(-n // k)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    op = case["op"]
    if op == "serve":
        return State(server=server(case["workers"]), items=serve_items(case, rng))
    ctx, k = context(), case["k"]
    off, nbr, ew, vw = host_graph(case, seed)
    graph = gp.Graph(ctx, off, nbr, ew, vw)
    if op == "partition":
        return State(graph=graph, k=k, seed=seed)
    if op == "coarsen":
        # Buffers for what comes back, long enough for any hierarchy of the
        # graph: the maps of all levels (about 2.2 n together), the coarsest graph.
        n, m = graph.n, graph.m
        return State(graph=graph, options=gp.coarsen_options(k, seed, **production(k)),
                     maps=np.zeros(3 * n, np.int32), off=np.zeros(n + 1, np.int32), vw=np.zeros(n, np.uint32),
                     nbr=np.zeros(size(case)[1], np.int32), ew=np.zeros(size(case)[1], np.uint32))
    if op == "uncoarsen":
        hierarchy = gp.Hierarchy(ctx, graph, gp.coarsen_options(k, seed, **production(k)))
        coarsest = hierarchy.graph_at(hierarchy.levels - 1)
        labels = gp.initial_partition_host(*coarsest, k, IMBALANCE, seed)
        return State(graph=graph, hierarchy=hierarchy, labels=labels, options=gp.refine_options(k, IMBALANCE))
    if op == "repartition":
        labels, _ = graph.partition(k, IMBALANCE, seed)
        u, v = new_edges(off, nbr, case["changes"], rng)
        return State(graph=graph, labels=labels, u=u, v=v, add=np.ones(len(u), np.uint8),
                     drop=np.zeros(len(u), np.uint8), options=gp.refine_options(k, IMBALANCE))
    # A candidate partition as a caller has it: blocks of neighbouring
    # vertices, one in eight vertices moved elsewhere.
    n = len(off) - 1
    labels = (np.arange(n, dtype=np.int64) * k // n).astype(np.int32)
    moved = rng.random(n) < 0.125
    labels[moved] = rng.integers(0, k, int(moved.sum()), dtype=np.int32)
    return State(graph=graph, k=k, labels=torch.from_numpy(labels).cuda())


def production(k):
    """The command-line tool's schedule: cluster sizes by the part count."""
    factor = max(64, -(-512 // k)) if k <= 8 else max(2, -(-32 // k))
    return dict(cluster_size_factor=factor, pack_isolated=1, progressive=int(k >= 16))


def run(state):
    kept = state.kept
    if "items" in kept:
        tickets = [kept["server"].submit(item) for item in kept["items"]]
        stats = [kept["server"].wait(t) for t in tickets]
        return {"labels": [item.labels for item in kept["items"]], "cuts": [s["final_cut"] for s in stats]}
    graph = kept["graph"]
    if "u" in kept:
        grown = gp.apply_delta(graph.ctx, graph.h, kept["u"], kept["v"], kept["add"])
        labels, stats = graph.refine(kept["labels"], kept["options"])
        back = gp.apply_delta(graph.ctx, graph.h, kept["u"], kept["v"], kept["drop"])
        return {"labels": labels, "cut": stats["final_cut"], "entries": [grown, back]}
    if "hierarchy" in kept:
        labels, cut, loads, _ = kept["hierarchy"].uncoarsen(kept["labels"], kept["options"])
        return {"labels": labels, "cut": cut, "loads": loads.astype(np.int64)}
    if "labels" in kept:
        cut, loads = graph.edge_cut(kept["labels"].data_ptr(), kept["k"])
        return {"cut": cut, "loads": loads.astype(np.int64)}
    if "options" in kept:
        hierarchy = gp.Hierarchy(graph.ctx, graph, kept["options"])
        last, at = hierarchy.levels - 1, 0
        for level in range(last):
            fine_to_coarse = hierarchy.map(level)
            kept["maps"][at:at + len(fine_to_coarse)] = fine_to_coarse
            at += len(fine_to_coarse)
        for name, values in zip(("off", "nbr", "ew", "vw"), hierarchy.graph_at(last)):
            kept[name][:len(values)] = values
        hierarchy.close()
        return {name: kept[name] for name in ("maps", "off", "nbr", "ew", "vw")}
    labels, stats = graph.partition(kept["k"], IMBALANCE, kept["seed"])
    return {"labels": labels, "cut": stats["final_cut"], "heaviest": stats["max_part_weight"]}


# ------------------------------------------------------------ what it takes
def size(case):
    """(vertices, entries, bytes a stored entry takes) of a case's graph."""
    kind = case["graph"]
    if kind == "grid":
        r, c = case["rows"], case["cols"]
        return r * c, 2 * (r * (c - 1) + c * (r - 1)), 4
    if kind == "mesh":
        return case["n"], 8 * case["n"], 4
    if kind == "rmat":
        n = 1 << case["scale"]
        return n, int(R_MAT_KEPT * 2 * case["degree"] * n), 4
    return case["n"], int(11.5 * case["n"]), 8


def work(case):
    """Bytes of the inputs read once and the outputs written once; the work
    is whole numbers, so the operations are one per entry visited."""
    op = case["op"]
    if op == "serve":
        # mean of sizes spread over their logarithm, mean degree about 12
        n = case["count"] * (case["largest"] - 1024) / math.log(case["largest"] / 1024)
        return {"bytes": n * (4 + 4 + 12 * 4), "flops": n * 12}
    n, m, entry = size(case)
    graph = 4 * (n + 1) + entry * m + (4 * n if entry == 8 else 0)
    if op == "coarsen":
        # the maps of all levels, each about half as long as the one before
        return {"bytes": graph + 2 * 4 * n, "flops": m}
    if op == "uncoarsen":
        # the graphs and maps of all levels, about twice the finest
        return {"bytes": 2 * (graph + 4 * n) + 4 * n, "flops": 2 * m}
    if op == "repartition":
        # both changes read and write the graph once, the refinement reads it
        return {"bytes": 5 * graph + 2 * 4 * n + 2 * 9 * case["changes"], "flops": 3 * m}
    return {"bytes": graph + 4 * n, "flops": m}


def tolerance(case):
    """Labels, maps, cuts and loads are whole numbers of a deterministic
    schedule: the same whatever the kernels."""
    return "exact"


def exact(case, seed):
    """Cut and loads recounted; a partition has no value but the one that the
    schedule gives."""
    if case["op"] != "edge_cut":
        return None
    off, nbr, ew, vw = host_graph(case, seed)
    labels = prepare(case, seed)["labels"].cpu().numpy()
    rows = np.repeat(np.arange(len(off) - 1), np.diff(off))
    weight = np.ones(len(nbr), np.int64) if ew is None else ew.astype(np.int64)
    cut = int(weight[labels[rows] != labels[nbr]].sum()) // 2
    mass = np.ones(len(labels), np.int64) if vw is None else vw.astype(np.int64)
    loads = np.zeros(case["k"], np.int64)
    np.add.at(loads, labels, mass)
    return {"cut": cut, "loads": loads}
