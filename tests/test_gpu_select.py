"""GPU: rebalance iterations against the oracle, at the sizes where their item counts and
paths change: small levels (both selections in one workgroup) and larger ones (slices of
the candidates, then one workgroup for the destinations).

Refinement starts from shuffled labels, which takes many LP rounds and rebalance
iterations with crowded boundary buckets. Labels, cuts and round counts are whole
numbers and must be equal.
"""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 1, 4 and 16 vertices per thread up to 1024, 4096 and 16384 vertices; above, the
# candidate lists
SIDES = [(3, 7), (32, 32), (25, 41), (64, 64), (17, 241), (128, 128), (5, 3277)]


@pytest.mark.parametrize("weights", ["unit", "wide", "with_zeros"])
@pytest.mark.parametrize("k", [2, 7, 32])
@pytest.mark.parametrize("sides", SIDES)
def test_small_level_rebalance_matches_oracle(hx, oracle, sides, k, weights):
    """wide: part weights beyond 32 bits, so the selection's histogram is 64 bits
    wide and, for k = 32, summed in two windows of parts."""
    if hx.device_count() < 1:
        pytest.skip("no GPU")
    n = sides[0] * sides[1]
    if n < 4 * k:
        pytest.skip("fewer than four vertices per part")
    print(f"case select sides={sides} k={k} weights={weights}", flush=True)
    indptr, indices = hx.generate_grid2d(*sides)
    rng = np.random.default_rng(n + k)
    ratio = 1.03 if n >= 64 * k else 1.3
    vw = None
    if weights == "wide":
        vw = (np.uint64(1) << np.uint64(33)) + rng.integers(0, 1 << 20, n).astype(np.uint64)
    elif weights == "with_zeros":
        vw = rng.integers(0, 3, n).astype(np.uint64)
        ratio = 1.6
    start = (rng.permutation(n) % k).astype(np.int32)
    og = oracle.Graph(indptr, indices.astype(np.int32), vertex_weights=vw)
    loads = oracle.part_weights(og, start, k)
    assert max(loads) <= oracle.partition_capacity(int(sum(loads)), k, ratio)
    expect, st = oracle.refine(og, start, k, ratio)
    g = hx.Graph(indptr, indices, "big" if weights == "wide" else "standard", vertex_weights=vw)
    labels, rep = g.refine(start, k, ratio)
    assert rep["rounds"] == st.rounds and rep["admission_iterations"] == st.admission_iterations
    assert rep["final_cut"] == st.final_cut
    assert np.array_equal(labels, expect)


# above 16384 vertices; 257 slices' worth of vertices; candidate tiles of 32 vertices per thread
@pytest.mark.parametrize("weights", ["unit", "wide"])
@pytest.mark.parametrize("k", [3, 32])
@pytest.mark.parametrize("sides", [(129, 130), (512, 514), (1449, 1450)])
def test_large_level_rebalance_matches_oracle(hx, oracle, sides, k, weights):
    if hx.device_count() < 1:
        pytest.skip("no GPU")
    n = sides[0] * sides[1]
    print(f"case large select sides={sides} k={k} weights={weights}", flush=True)
    indptr, indices = hx.generate_grid2d(*sides)
    rng = np.random.default_rng(n + k)
    vw = None
    if weights == "wide":
        vw = (np.uint64(1) << np.uint64(33)) + rng.integers(0, 1 << 20, n).astype(np.uint64)
    start = (rng.permutation(n) % k).astype(np.int32)
    og = oracle.Graph(indptr, indices.astype(np.int32), vertex_weights=vw)
    expect, st = oracle.refine(og, start, k, 1.005, 4, 4)
    assert st.admission_iterations > 0
    g = hx.Graph(indptr, indices, "big" if weights == "wide" else "standard", vertex_weights=vw)
    labels, rep = g.refine(start, k, 1.005, 4, 4)
    assert rep["rounds"] == st.rounds and rep["admission_iterations"] == st.admission_iterations
    assert rep["final_cut"] == st.final_cut
    assert np.array_equal(labels, expect)
