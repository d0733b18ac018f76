"""GPU: refinement of a graph that is on the device already refuses what the reference's
host form refuses (src/refine.cu:259-343 of the reference), with the same kind of error
and the caller's labels untouched."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _refused(hx, g, labels, k, ratio):
    given = labels.copy()
    with pytest.raises(hx.GpartError) as e:
        g.refine(labels, k, ratio)
    assert np.array_equal(labels, given)
    return e.value.kind, str(e.value)


def test_refine_refuses_what_the_host_form_refuses(hx):
    if hx.device_count() < 1:
        pytest.skip("no GPU")
    indptr, indices = hx.generate_grid2d(8, 8)
    balanced = (np.arange(64) % 4).astype(np.int32)
    g = hx.Graph(indptr, indices)
    for bad in (-1, 4, 2**31 - 1):
        labels = balanced.copy()
        labels[63] = bad
        assert _refused(hx, g, labels, 4, 1.03) == ("invalid_argument", "refinement partition has an invalid part id")
    lopsided = np.minimum(balanced, 1).astype(np.int32)
    assert _refused(hx, g, lopsided, 4, 1.03) == ("invalid_argument", "initial refinement partition is imbalanced")
    for k, ratio in ((1, 1.03), (33, 1.03), (4, 0.5), (4, float("nan"))):
        assert _refused(hx, g, balanced.copy(), k, ratio) == ("invalid_argument", "invalid refinement options")
    # a vertex weight sum past 64 bits, and an invalid part met before or after it
    heavy = hx.Graph(indptr, indices, "big", vertex_weights=np.full(64, 1 << 60, np.uint64))
    assert _refused(hx, heavy, balanced.copy(), 4, 1.03)[0] == "overflow_error"
    labels = balanced.copy()
    labels[0] = 9
    assert _refused(hx, heavy, labels, 4, 1.03)[0] == "invalid_argument"
    labels = balanced.copy()
    labels[63] = 9
    assert _refused(hx, heavy, labels, 4, 1.03)[0] == "overflow_error"


def test_refine_keeps_the_resident_graph(hx, oracle):
    if hx.device_count() < 1:
        pytest.skip("no GPU")
    indptr, indices = hx.generate_grid2d(40, 41)
    g = hx.Graph(indptr, indices)
    before = g.arrays()
    start = (np.random.default_rng(3).permutation(g.n) % 5).astype(np.int32)
    expect, _ = oracle.refine(oracle.Graph(indptr, indices.astype(np.int32)), start, 5, 1.05)
    for _ in range(2):
        labels, rep = g.refine(start, 5, 1.05)
        assert np.array_equal(labels, expect) and rep["final_cut"] == g.cut(labels)
    for a, b in zip(before, g.arrays()):
        assert np.array_equal(a, b)
