"""GPU: refinement of dense levels, whose connectivity rows are summed from the CSR
when a round reads them, against the oracle.

The graphs cover what the form distinguishes: rows of every degree class, hub rows of
several chunks, vertex states of a byte and of half a byte (k <= 8 on levels above
131,072 vertices) in LDS and of a byte in memory (above, from k = 9 on, or above 262,144
vertices), both widths, unit and larger entry weights, and the neighbours of a
mover that move too. Labels, cuts and round counts are whole numbers and must be equal.
"""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _csr(src, dst, n):
    """Symmetric CSR without duplicates or self loops."""
    a, b = np.concatenate([src, dst]), np.concatenate([dst, src])
    keep = a != b
    key = np.unique(a[keep].astype(np.int64) * n + b[keep])
    indptr = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(key // n, minlength=n), out=indptr[1:])
    return indptr, key % n


def random_graph(hx, n, degree):
    rng = np.random.default_rng(n)
    return _csr(rng.integers(0, n, n * degree // 2), rng.integers(0, n, n * degree // 2), n)


def hub_graph(hx, n, hubs):
    """Every hub adjacent to most vertices, the rest sparse: rows of several chunks."""
    rng = np.random.default_rng(hubs)
    src = [np.full(n * 3 // 4, h) for h in range(hubs)] + [rng.integers(0, n, 2 * n)]
    dst = [rng.choice(n, n * 3 // 4, replace=False) for _ in range(hubs)] + [rng.integers(0, n, 2 * n)]
    return _csr(np.concatenate(src), np.concatenate(dst), n)


GRAPHS = {
    "rmat10": lambda hx: hx.generate_rmat(10, 32),
    "rmat13": lambda hx: hx.generate_rmat(13, 32),
    "hubs12001": lambda hx: hub_graph(hx, 12_001, 24),
    "hubs20011": lambda hx: hub_graph(hx, 20_011, 20),
    "byte131072": lambda hx: random_graph(hx, 131_072, 26),
    "random131073": lambda hx: random_graph(hx, 131_073, 26),
    "memory262145": lambda hx: random_graph(hx, 262_145, 26),
    "hubs140001": lambda hx: hub_graph(hx, 140_001, 16),
}


@pytest.mark.parametrize("name,k,width,weighted", [
    ("rmat10", 2, "standard", False), ("rmat10", 32, "big", True), ("rmat13", 8, "standard", True),
    ("rmat13", 31, "standard", False), ("hubs12001", 8, "standard", True), ("hubs12001", 32, "big", False),
    ("hubs20011", 5, "big", True), ("hubs20011", 32, "standard", False), ("byte131072", 9, "standard", False),
    ("random131073", 8, "standard", True), ("random131073", 7, "big", False),
    ("random131073", 9, "standard", True), ("random131073", 32, "big", False), ("memory262145", 8, "big", True),
    ("hubs140001", 9, "big", False), ("hubs140001", 32, "standard", True),
])
def test_dense_refinement_matches_oracle(hx, oracle, name, k, width, weighted):
    if hx.device_count() < 1:
        pytest.skip("no GPU")
    print(f"case rows graph={name} k={k} width={width} weighted={weighted}", flush=True)
    indptr, indices = GRAPHS[name](hx)
    n, m = len(indptr) - 1, len(indices)
    assert m >= 24 * n
    ew = None
    if weighted:
        salt = np.random.default_rng(k).integers(1, 1 << 20, n).astype(np.uint64)
        src = np.repeat(np.arange(n), np.diff(indptr))
        ew = np.uint64(1) + (salt[src] ^ salt[indices]) % np.uint64(9)
    start = (np.random.default_rng(k).permutation(n) % k).astype(np.int32)
    og = oracle.Graph(indptr, indices.astype(np.int32), edge_weights=ew)
    expect, st = oracle.refine(og, start, k, 1.03, 6, 3)
    assert st.accepted > 0 and st.admission_iterations > 0
    g = hx.Graph(indptr, indices, width, edge_weights=ew)
    labels, rep = g.refine(start, k, 1.03, 6, 3)
    assert rep["rounds"] == st.rounds and rep["admission_iterations"] == st.admission_iterations
    assert rep["final_cut"] == st.final_cut
    assert np.array_equal(labels, expect)
    # the strict checks recount the cut and compare the rows of every round
    strict, _ = g.refine(start, k, 1.03, 6, 3, verify=True)
    assert np.array_equal(strict, expect)
