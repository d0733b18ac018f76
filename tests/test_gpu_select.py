"""GPU: rebalance iterations against the oracle, at the sizes where their item counts and
paths change: small levels (both selections in one workgroup) and larger ones (slices of
the candidates for the sources; one workgroup, or passes over the slices, for the
destinations).

Refinement starts from shuffled labels, which takes many LP rounds and rebalance
iterations with crowded boundary buckets. Labels, cuts and round counts are whole
numbers and must be equal.
"""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_refine_rows import random_graph

pytestmark = pytest.mark.gpu

# 1, 4 and 16 vertices per thread up to 1024, 4096 and 16384 vertices; above, the
# candidate lists
SIDES = [(3, 7), (32, 32), (25, 41), (64, 64), (17, 241), (128, 128), (5, 3277)]
SMALL = [(sides, k) for sides in SIDES for k in (2, 7, 32) if sides[0] * sides[1] >= 4 * k]


@pytest.mark.parametrize("weights", ["unit", "wide", "with_zeros"])
@pytest.mark.parametrize("sides,k", SMALL)
def test_small_level_rebalance_matches_oracle(hx, oracle, sides, k, weights):
    """wide: part weights beyond 32 bits, so the selection's histogram is 64 bits
    wide and, for k = 32, summed in two windows of parts."""
    if hx.device_count() < 1:
        pytest.skip("no GPU")
    n = sides[0] * sides[1]
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


@pytest.fixture
def few_leaving(hx):
    yield hx.set_refine_few_leaving
    hx.set_refine_few_leaving()


def shuffled(n, k):
    return (np.random.default_rng(n + k).permutation(n) % k).astype(np.int32)


def compare(hx, oracle, indptr, indices, vw, k, width, ratio, start, rounds=(4, 4)):
    """Refinement of the labels, equal to the oracle's; the large iterations by form."""
    og = oracle.Graph(indptr, indices.astype(np.int32), vertex_weights=vw)
    expect, st = oracle.refine(og, start, k, ratio, *rounds)
    assert st.admission_iterations > 0
    g = hx.Graph(indptr, indices, width, vertex_weights=vw)
    before = hx.refine_selection_stats()
    labels, rep = g.refine(start, k, ratio, *rounds)
    assert rep["rounds"] == st.rounds and rep["admission_iterations"] == st.admission_iterations
    assert rep["final_cut"] == st.final_cut
    assert np.array_equal(labels, expect)
    after = hx.refine_selection_stats()
    counts = {form: after[form] - before[form] for form in after}
    assert counts["single"] + counts["slices"] == st.admission_iterations
    return counts


# above 16384 vertices; 257 slices' worth of vertices; candidate tiles of 32 vertices per thread
@pytest.mark.parametrize("form", ["single", "slices"])
@pytest.mark.parametrize("weights", ["unit", "wide"])
@pytest.mark.parametrize("k", [3, 32])
@pytest.mark.parametrize("sides", [(129, 130), (512, 514), (1449, 1450)])
def test_large_level_rebalance_matches_oracle(hx, oracle, few_leaving, sides, k, weights, form):
    if hx.device_count() < 1:
        pytest.skip("no GPU")
    n = sides[0] * sides[1]
    print(f"case large select sides={sides} k={k} weights={weights} form={form}", flush=True)
    indptr, indices = hx.generate_grid2d(*sides)
    vw = None
    if weights == "wide":
        vw = (np.uint64(1) << np.uint64(33)) + np.random.default_rng(n + k).integers(0, 1 << 20, n).astype(np.uint64)
    few_leaving(1 << 28 if form == "single" else -1)
    counts = compare(hx, oracle, indptr, indices, vw, k, "big" if weights == "wide" else "standard", 1.005,
                     shuffled(n, k))
    assert counts[form] > 0 and sum(counts.values()) == counts[form]


@pytest.mark.parametrize("width", ["standard", "big"])
@pytest.mark.parametrize("dense", [False, True])
def test_more_leave_than_expected(hx, oracle, few_leaving, dense, width):
    """A few vertices hold most of the weight, so the leaving ones, all light, are far more
    than their weight's share of the vertices: the workgroup refuses and the iteration
    runs again. dense: levels whose rows are summed where they are read."""
    if hx.device_count() < 1:
        pytest.skip("no GPU")
    print(f"case refused selection dense={dense} width={width}", flush=True)
    indptr, indices = random_graph(hx, 20_001, 26) if dense else hx.generate_grid2d(150, 151)
    n, k = len(indptr) - 1, 3
    vw = np.ones(n, np.uint64)
    start = shuffled(n, k)
    heavy = np.arange(5 * k) * 7
    vw[heavy], start[heavy] = 1_000_000, np.arange(5 * k) % k
    few_leaving(4)
    counts = compare(hx, oracle, indptr, indices, vw, k, width, 1.0001, start)
    assert counts["refused"] > 0
