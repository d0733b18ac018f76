"""The work a user of the partitioner has it do, as measurable cases.

A case is a dict of plain values; "op" names the public call it makes:

  partition  Graph.partition on a graph resident on the GPU, labels to the host: the
             call of the partition tool and of every binding
  upload     host int64 CSR with weights -> Graph -> partition, as a program does whose
             weighted graph lives in host memory
  batch      partition_batch over several graphs (the graph mix)
  refine     Graph.refine of labels that a program already holds (repartitioning)
  aggregate  Graph.aggregate, one level of clustering as an entry point of its own
  check      Graph.verify and Graph.analyze of a labelling (the two checking tools)
  initial    Graph.initial_partition of a coarse graph, with its coordinates

Graphs are lattices (2D grid, 3D mesh) and R-MAT graphs (0.57, 0.19, 0.19), the
families of the benchmark and its graph mix. Every result is a whole number or, for
the coordinates and ratios, fixed by a stated order of FP64 operations, so every
comparison is exact.
"""
from __future__ import annotations

import math

import numpy as np

import horkxg_amd as hx
from horkxg_amd.workloads import mix_spec

hx.set_log(False)  # no progress lines on stdout


def _case(name, op, kind, size, k, width="standard", mode="batched_fp64", **more):
    return dict(name=name, op=op, kind=kind, a=size[0], b=size[1], c=size[2] if len(size) > 2 else 1, k=k,
                width=width, mode=mode, **more)


def listed():
    return [
        # the smallest call: a graph that coarsens in a level or two, launches and host waits count
        _case("grid64_k4", "partition", "grid2d", (64, 64), 4),
        # the benchmark's small configuration
        _case("grid256_k4", "partition", "grid2d", (256, 256), 4),
        # the benchmark's default: a large regular mesh into the most parts
        _case("mesh128_k32", "partition", "mesh3d", (128, 128, 128), 32),
        # a social-network-like graph of ordinary size, FP32 bisection as the R-MAT configurations run it
        _case("rmat18_k8", "partition", "rmat", (18, 16), 8, mode="batched_fp32"),
        # the benchmark's large standard-width configuration
        _case("rmat22_k8", "partition", "rmat", (22, 16), 8, mode="batched_fp32"),
        # 64-bit offsets and weights, the largest graph here: stands for the scale-26 configuration
        _case("rmat24_k32_big", "partition", "rmat", (24, 16), 32, "big", "batched_fp32"),
        # a weighted mesh with odd sides and a part count that is no power of two, from host arrays
        _case("wmesh_k12_upload_big", "upload", "mesh3d", (47, 53, 61), 12, "big"),
        # sixteen small and middling graphs of the mix, one call
        _case("mix16_batch", "batch", "mix", (0, 16), 0, mode="batched_fp32", max_n=200_000),
        # labels that a program holds already, disturbed, brought back to a good cut
        _case("refine_mesh96_k16", "refine", "mesh3d", (96, 97, 95), 16),
        # one clustering of a skewed graph, its map and cluster weights
        _case("aggregate_rmat19_k16", "aggregate", "rmat", (19, 16), 16),
        # the checking tools' calls
        _case("check_rmat20_k32", "check", "rmat", (20, 16), 32),
        # the initial partition of a coarse weighted graph as an entry point of its own
        _case("initial_mesh_k32", "initial", "mesh3d", (23, 19, 17), 32, "big"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _lattice(rng, low, high):
    n = _log_int(rng, low, high)
    if rng.random() < 0.5:
        a = max(3, int(math.sqrt(n) * rng.uniform(0.6, 1.6)))
        return "grid2d", (a, max(3, n // a))
    side = n ** (1.0 / 3.0)
    a = max(3, int(side * rng.uniform(0.7, 1.4)))
    b = max(3, int(side * rng.uniform(0.7, 1.4)))
    return "mesh3d", (a, b, max(3, n // (a * b)))


def _any_graph(rng, low, high, rmat_high):
    if rng.random() < 0.5:
        return _lattice(rng, low, high)
    scale = rng.randint(int(math.log2(low)), rmat_high)
    return "rmat", (scale, rng.randint(5, 16))


def _parts(rng, n):
    return rng.randint(2, max(2, min(32, n // 1024)))


def draw(rng):
    op = rng.choice(["partition"] * 6 + ["upload", "batch", "refine", "aggregate", "check", "initial"])
    width = rng.choice(["standard", "standard", "big"])
    mode = rng.choice(["batched_fp64", "batched_fp32", "plain_fp64"])
    if op == "partition":
        kind, size = _any_graph(rng, 4096, 2_500_000, 22)
    elif op == "upload":
        kind, size = _lattice(rng, 4096, 200_000)
    elif op == "batch":
        first, count = rng.randint(0, 200), rng.randint(3, 16)
        return dict(op="batch", kind="mix", a=first, b=count, c=1, k=0, width="standard", mode="batched_fp32",
                    max_n=_log_int(rng, 20_000, 250_000))
    elif op == "refine":
        kind, size = _lattice(rng, 8192, 1_000_000)
    elif op == "aggregate":
        kind, size = _any_graph(rng, 4096, 2_000_000, 20)
    elif op == "check":
        kind, size = _any_graph(rng, 4096, 1_000_000, 20)
    else:
        kind, size = _lattice(rng, 1500, 16_000)
    n = 1 << size[0] if kind == "rmat" else math.prod(size)
    c = _case("", op, kind, size, _parts(rng, n), width, mode)
    del c["name"]
    return c


def _size(case):
    """(vertices, directed entries); an R-MAT graph keeps about nine tenths of its samples."""
    a, b, c = case["a"], case["b"], case["c"]
    if case["kind"] == "rmat":
        return 1 << a, int(1.8 * b * (1 << a))
    return a * b * c, 2 * ((a - 1) * b * c + a * (b - 1) * c + a * b * (c - 1))


def _mix(case):
    return [mix_spec(case["a"] + i, max_n=case["max_n"]) for i in range(case["b"])]


def _lattice_rows(kind, size, width):
    if kind == "grid2d":
        return hx.Graph.generate_grid2d(size[0], size[1], width=width)
    return hx.Graph.generate_mesh3d(*size, width=width)


def _resident(case, seed):
    if case["kind"] == "rmat":
        return hx.Graph.generate_rmat(case["a"], case["b"], 0.57, 0.19, 0.19, seed, width=case["width"])
    return _lattice_rows(case["kind"], (case["a"], case["b"], case["c"]), case["width"])


def _weights(indptr, indices, seed):
    """Symmetric edge weights in [1, 8] and vertex weights in [1, 3]."""
    rng = np.random.default_rng(seed)
    n = len(indptr) - 1
    src = np.repeat(np.arange(n, dtype=np.int64), np.diff(indptr))
    salt = rng.integers(1, 1 << 30, n).astype(np.uint64)
    ew = np.uint64(1) + ((salt[src] ^ salt[indices]) >> np.uint64(7)) % np.uint64(8)
    vw = rng.integers(1, 4, n).astype(np.uint64)
    return ew, vw


def _host_lattice(case):
    if case["kind"] == "grid2d":
        return hx.generate_grid2d(case["a"], case["b"])
    return hx.generate_mesh3d(case["a"], case["b"], case["c"])


def prepare(case, seed):
    op, k = case["op"], case["k"]
    state = dict(case=case, seed=seed % (1 << 31))
    if op == "batch":
        state["specs"] = specs = _mix(case)
        state["seeds"] = [(seed * 1000 + s["seed"]) % (1 << 31) for s in specs]
        state["graphs"] = []
        for s, graph_seed in zip(specs, state["seeds"]):
            if s["kind"] == "rmat":
                g = hx.Graph.generate_rmat(s["size"][0], s["size"][1], 0.57, 0.19, 0.19, graph_seed)
            else:
                g = _lattice_rows(s["kind"], s["size"], "standard")
            state["graphs"].append(g)
    elif op in ("upload", "initial"):
        indptr, indices = _host_lattice(case)
        ew, vw = _weights(indptr, indices, seed)
        if op == "upload":
            state["arrays"] = (indptr, indices, ew, vw)
        else:
            state["graph"] = hx.Graph(indptr, indices, case["width"], ew, vw)
    else:
        state["graph"] = g = _resident(case, seed)
        rng = np.random.default_rng(seed)
        if op == "refine":
            # slabs in id order, a tenth of the vertices with shuffled labels: loads stay as they were
            labels = (np.arange(g.n, dtype=np.int64) * k // g.n).astype(np.int32)
            moved = rng.choice(g.n, g.n // 10, replace=False)
            labels[moved] = labels[rng.permutation(moved)]
            state["labels"] = labels
        elif op == "check":
            state["labels"] = rng.integers(0, k, g.n).astype(np.int32)
    return state


REPORT = ("final_cut", "max_part_weight", "capacity", "initial_cut", "coarsest_vertices", "levels", "refined_levels")
REFINE = ("rounds", "admission_iterations", "admission_fallbacks", "proposals", "accepted", "initial_cut", "final_cut",
          "final_max_part_weight")
VERIFY = ("vertices", "undirected_edges", "cut", "max_load", "capacity")
COUNTS = ("parts", "vertices", "directed_edges", "edge_cut", "weighted_edge_cut", "max_local_cut",
          "weighted_max_local_cut", "min_vertices", "max_vertices", "min_edge_set", "max_edge_set")


def _whole(report, names):
    return np.array([int(report[x]) for x in names], np.int64)


def run(state):
    case, seed = state["case"], state["seed"]
    op, k, mode = case["op"], case["k"], case["mode"]
    if op == "partition":
        labels, rep = state["graph"].partition(k, 1.03, seed, spectral_mode=mode)
        return [labels, _whole(rep, REPORT)]
    if op == "upload":
        indptr, indices, ew, vw = state["arrays"]
        g = hx.Graph(indptr, indices, case["width"], ew, vw)
        labels, rep = g.partition(k, 1.03, seed, spectral_mode=mode)
        return [labels, _whole(rep, REPORT)]
    if op == "batch":
        labels, reps, _ = hx.partition_batch(state["graphs"], [s["k"] for s in state["specs"]],
                                             seeds=state["seeds"], spectral_mode=mode)
        return list(labels) + [_whole(r, REPORT) for r in reps]
    if op == "refine":
        labels, rep = state["graph"].refine(state["labels"], k)
        return [labels, _whole(rep, REFINE)]
    if op == "aggregate":
        mapping, weights, coarse, capacity, heaviest = state["graph"].aggregate(k, seed)
        padded = np.zeros(len(mapping), np.uint64)  # one shape whatever the number of clusters
        padded[:coarse] = weights
        return [mapping, padded, np.array([coarse, capacity, heaviest], np.int64)]
    if op == "check":
        g, labels = state["graph"], state["labels"]
        ver = g.verify(labels, k, "1.03")
        ana = g.analyze(labels, k)
        return [_whole(ver, VERIFY), np.array(ver["loads"], np.int64), _whole(ana, COUNTS)] + \
            [np.asarray(v) for _, v in sorted(ana["per_part"].items())]
    labels, coords = state["graph"].initial_partition(k, 1.03, seed, spectral_mode=mode, with_coords=True)
    return [labels, coords]


def work(case):
    """Bytes of one pass: the graph read once in its own width, labels written (or read) once."""
    if case["op"] == "batch":
        total = 0
        for s in _mix(case):
            size = tuple(s["size"]) + (1,)
            n, m = _size(dict(kind=s["kind"], a=size[0], b=size[1], c=size[2]))
            total += 12 * n + 8 * m
        return {"bytes": total, "flops": 0}
    n, m = _size(case)
    wide = 8 if case["width"] == "big" else 4
    csr = wide * (n + 1) + (4 + wide) * m + wide * n
    if case["op"] == "upload":  # int64 offsets and neighbours, 64-bit weights
        return {"bytes": 8 * (n + 1) + 16 * m + 8 * n + 4 * n, "flops": 0}
    if case["op"] == "aggregate":  # the map, and about half as many cluster weights
        return {"bytes": csr + 8 * n, "flops": 0}
    if case["op"] == "check":  # verify and analyze each read the graph and the labels
        return {"bytes": 2 * (csr + 4 * n), "flops": 0}
    if case["op"] == "initial":  # 64 diffusion steps, a multiply-add per entry, at every level of the recursion
        return {"bytes": csr + 12 * n, "flops": 128 * m * max(1, math.ceil(math.log2(case["k"])))}
    return {"bytes": csr + (8 if case["op"] == "refine" else 4) * n, "flops": 0}


def tolerance(case):
    """Every output is a whole number, or FP64 coordinates with a stated order of operations."""
    return "exact"


def exact(case, seed):
    """The checking tools' counters in numpy; the partitions themselves are the outcome of a
    heuristic with no closed form."""
    if case["op"] != "check":
        return None
    state = prepare(case, seed)
    off, adj, ew, _ = state["graph"].arrays()
    lab, k, n = state["labels"].astype(np.int64), case["k"], state["graph"].n
    src = np.repeat(np.arange(n, dtype=np.int64), np.diff(off))
    ps, pd = lab[src], lab[adj]
    cut = ps != pd
    loads = np.bincount(lab, minlength=k)
    directed, nonloop = int(cut.sum()), int((src != adj).sum())
    capacity = 103 * n // (100 * k)
    verify = np.array([n, nonloop // 2, directed // 2, loads.max(), capacity], np.int64)
    internal = np.bincount(ps[~cut], minlength=k)
    outgoing, incoming = np.bincount(ps[cut], minlength=k), np.bincount(pd[cut], minlength=k)
    local, edge_set = outgoing + incoming, internal + outgoing + incoming
    # unit edge weights: the weighted counters are the plain ones
    counts = np.array([k, n, len(adj), directed, directed, local.max(), local.max(), loads.min(), loads.max(),
                       edge_set.min(), edge_set.max()], np.int64)
    per_part = dict(vertices=loads, internal=internal, outgoing=outgoing, incoming=incoming,
                    weighted_internal=internal, weighted_outgoing=outgoing, weighted_incoming=incoming)
    return [verify, loads.astype(np.int64), counts] + [v.astype(np.int64) for _, v in sorted(per_part.items())]
