"""A depth of small sparse bisection tasks in one launch (hip/initial.hip, depth_solo_kernel).

A workgroup does a task's start, 64 steps and split, where every task of the depth has at
most 416 rows of 64 slots, rows of at most 96 and weights below 2^52; else the depth takes
its 66 launches. FP64 labels and coordinates must be
bit-identical to the oracle's recursive bisection (src/initial_partition_gpu.cu:170-276),
FP32 ones to the task queue's, which sums the same terms in the same order.
"""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def lattice(n, half_degree, weight=lambda a, b: 1 + (a * 7 + b) % 5, hubs=(), hub_degree=0):
    """A ring whose vertices meet their next `half_degree` ones; hubs meet `hub_degree` more."""
    edges = {}
    for v in range(n):
        for d in range(1, half_degree + 1):
            a, b = sorted((v, (v + d) % n))
            if a != b:
                edges[a, b] = weight(a, b)
    for h in hubs:
        for d in range(hub_degree):
            a, b = sorted((h, (h + 3 + 17 * d) % n))
            if a != b:
                edges[a, b] = weight(a, b)
    rows = [[] for _ in range(n)]
    for (a, b), w in edges.items():
        rows[a].append((b, w))
        rows[b].append((a, w))
    off = np.zeros(n + 1, np.int64)
    off[1:] = np.cumsum([len(r) for r in rows])
    adj = np.array([u for r in rows for u, _ in sorted(r)], np.int32)
    ew = np.array([w for r in rows for _, w in sorted(r)], np.uint64)
    vw = (1 + np.arange(n) % 3).astype(np.uint64)
    return off, adj, ew, vw


CASES = {
    # sizes at the edges of a block of 8, a wave, the workgroup and the largest task
    "n9": (lattice, (9, 1), "standard"),
    "n64": (lattice, (64, 2), "standard"),
    "n65_big": (lattice, (65, 3), "big"),
    "n1023": (lattice, (1023, 2), "standard"),
    "n1025": (lattice, (1025, 1), "big"),
    "n4096": (lattice, (4096, 2), "standard"),
    # roots too large for a depth: steps of one launch up to 8192 vertices, of three above
    "n4097": (lattice, (4097, 2), "big"),
    "n8192": (lattice, (8192, 1), "standard"),
    "n8193": (lattice, (8193, 1), "standard"),
    # slots per row: 8, 12, 16, 24, 32, more than 32 terms
    "deg8": (lattice, (700, 4), "standard"),
    "deg12": (lattice, (700, 6), "standard"),
    "deg16": (lattice, (700, 8), "big"),
    "deg22": (lattice, (700, 11), "standard"),
    "deg30": (lattice, (540, 15), "big"),
    "deg34": (lattice, (470, 17), "standard"),
    "deg34_solo": (lattice, (200, 17), "standard"),
    # one long row per wave: more slots than the form takes
    "hubs": (lambda: lattice(4096, 1, hubs=range(5, 4096, 64), hub_degree=60), (), "standard"),
    # a row too long for the form
    "hub": (lambda: lattice(3000, 1, hubs=(700, 2100), hub_degree=900), (), "big"),
    # weights beyond a 4-byte slot, at its edge, at an 8-byte one's and beyond it
    "wide": (lambda: lattice(300, 3, weight=lambda a, b: 2**20 - 1 + (a + b) % 2), (), "standard"),
    "wide_big": (lambda: lattice(300, 3, weight=lambda a, b: 2**40 + a), (), "big"),
    "wide_edge": (lambda: lattice(300, 2, weight=lambda a, b: 2**52 - 1 - (a + b) % 2), (), "big"),
    "widest": (lambda: lattice(300, 2, weight=lambda a, b: 2**52 + a * 2**20), (), "big"),
}


@pytest.fixture
def no_queue(hx):
    saved = hx.spectral_queue_settings()
    yield
    hx.set_spectral_queue(saved["enabled"], saved["own_blocks"], saved["max_task"])


@pytest.mark.parametrize("name", list(CASES))
def test_solo_depths(hx, oracle, no_queue, name):
    make, args, width = CASES[name]
    off, adj, ew, vw = make(*args)
    g = hx.Graph(off, adj, width=width, edge_weights=ew, vertex_weights=vw)
    og = oracle.Graph(off, adj, ew, vw)
    for k in (2, 7):
        print(f"case solo {name} k={k} n={len(off) - 1} m={len(adj)}", flush=True)
        hx.set_spectral_queue(False)
        labels, coords = g.initial_partition(k, 1.2, 3, "batched_fp64", with_coords=True)
        ol, oc, _ = oracle.initial_partition(og, k, 1.2, 3, with_coords=True)
        assert np.array_equal(labels, ol), k
        assert np.array_equal(coords.view(np.uint64), oc.view(np.uint64)), k
        labels, coords = g.initial_partition(k, 1.2, 3, "batched_fp32", with_coords=True)
        hx.set_spectral_queue(True, 64, 4096)
        ql, qc = g.initial_partition(k, 1.2, 3, "batched_fp32", with_coords=True)
        assert np.array_equal(labels, ql), k
        assert np.array_equal(coords.view(np.uint64), qc.view(np.uint64)), k


# a row of 27 to 32 entries in each of 13 groups: 416 rows of slots, and 4 more for one more
# vertex; rows of 96 and of 98; weights of 52 and 53 bits
HUBS = dict(hubs=range(5, 832, 64), hub_degree=26)


@pytest.mark.parametrize("name,make,width,solo", [
    ("rows", lambda: lattice(832, 1, **HUBS), "standard", True),
    ("more rows", lambda: lattice(833, 1, **HUBS), "standard", False),
    ("width", lambda: lattice(160, 48), "big", True), ("wider", lambda: lattice(160, 49), "big", False),
    ("weights", lambda: lattice(300, 2, lambda a, b: 2**52 - 1), "big", True),
    ("heavier", lambda: lattice(300, 2, lambda a, b: 2**52), "big", False)])
def test_form_of_a_depth(hx, oracle, no_queue, name, make, width, solo):
    """A refused depth is launched in both forms; the results are the oracle's either way."""
    off, adj, ew, vw = make()
    print(f"case solo form {name} n={len(off) - 1} m={len(adj)}", flush=True)
    g = hx.Graph(off, adj, width=width, edge_weights=ew, vertex_weights=vw)
    ol, oc, _ = oracle.initial_partition(oracle.Graph(off, adj, ew, vw), 2, 1.2, 3, with_coords=True)
    hx.set_spectral_queue(False)
    hx.profile_reset()
    hx.profile_enable("spectral", True)
    try:
        labels, coords = g.initial_partition(2, 1.2, 3, "batched_fp64", with_coords=True)
        launches = hx.profile_read("spectral")["launches"]
    finally:
        hx.profile_enable("spectral", False)
    assert np.array_equal(labels, ol)
    assert np.array_equal(coords.view(np.uint64), oc.view(np.uint64))
    assert launches == (1 if solo else 2)


def test_skewed_graphs(hx, oracle, no_queue):
    """Coarse graphs with long rows, at whose depths some tasks suit the form and others do not."""
    for scale, factor in ((9, 4), (11, 8), (12, 8)):
        indptr, indices = hx.generate_rmat(scale, factor)
        print(f"case solo rmat scale={scale} m={len(indices)}", flush=True)
        g, og = hx.Graph(indptr, indices), oracle.Graph(indptr, indices.astype(np.int32))
        hx.set_spectral_queue(False)
        labels, coords = g.initial_partition(16, 1.2, 3, "batched_fp64", with_coords=True)
        ol, oc, _ = oracle.initial_partition(og, 16, 1.2, 3, with_coords=True)
        assert np.array_equal(labels, ol), scale
        assert np.array_equal(coords.view(np.uint64), oc.view(np.uint64)), scale
