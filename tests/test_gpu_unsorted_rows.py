"""GPU: graphs whose rows are not strictly ascending (unsorted, or with parallel entries).

gpart_record_bounds reports them (src/coarsen.cu:44-70): the first clustering round offers
a row's entries one by one only where no neighbour repeats, and sums parallel entries
otherwise. Hierarchies and labels are whole numbers and must equal the oracle's.
"""
from __future__ import annotations

import ctypes as C

import kat_graphs as K
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def multigraph(n, pairs, seed, shuffled):
    """Random pairs, a third of them listed up to four times; rows sorted or shuffled."""
    rng = np.random.default_rng(seed)
    a, b = rng.integers(0, n, pairs), rng.integers(0, n, pairs)
    w = rng.integers(1, 9, pairs)
    keep = a != b
    a, b, w = a[keep], b[keep], w[keep]
    times = np.where(rng.random(len(a)) < 1 / 3, rng.integers(2, 5, len(a)), 1)
    a, b, w = np.repeat(a, times), np.repeat(b, times), np.repeat(w, times)
    src, dst, ew = np.concatenate([a, b]), np.concatenate([b, a]), np.concatenate([w, w])
    order = np.lexsort((rng.random(len(src)) if shuffled else dst, src))
    indptr = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(src, minlength=n), out=indptr[1:])
    return dict(indptr=indptr, indices=dst[order], edge_weights=ew[order].astype(np.uint64),
                vertex_weights=np.ones(n, np.uint64))


GRAPHS = {
    "hub259": lambda: K.hub259(),
    "multi": lambda: multigraph(2000, 6000, 1, False),
    "shuffled": lambda: multigraph(2000, 6000, 2, True),
    # rows of every degree class: up to 8, up to 256 and above
    "dense": lambda: multigraph(400, 30_000, 3, False),
}


@pytest.fixture(scope="module", autouse=True)
def need_gpu(hx):
    if hx.device_count() < 1:
        pytest.skip("no GPU")


# a row of the low, medium and high degree class, beside rows of the other two
@pytest.mark.parametrize("row", [0, 1, 2])
@pytest.mark.parametrize("kind", ["sorted", "unsorted", "duplicated"])
@pytest.mark.parametrize("width", ["standard", "big"])
def test_record_bounds_report_unsorted_rows(hx, row, kind, width):
    print(f"case record bounds row={row} kind={kind} width={width}", flush=True)
    from horkxg_amd.device import DeviceArray, _check, _ctx, hip_lib

    n, degrees = 700, [7, 200, 600]
    adj = [np.arange(10, 10 + d) for d in degrees]
    if kind == "unsorted":
        adj[row][[-2, -1]] = adj[row][[-1, -2]]
    elif kind == "duplicated":
        adj[row][-1] = adj[row][-2]
    indptr = np.concatenate([[0], np.cumsum(degrees), np.full(n - 3, sum(degrees))]).astype(np.int64)
    ew = np.random.default_rng(row).integers(1, 1000, sum(degrees)).astype(np.uint64)
    g = hx.device.DeviceGraph(indptr, np.concatenate(adj), ew, width=width)
    call = hip_lib().gpart_record_bounds
    call.argtypes = [C.c_void_p] * 5
    bounds = DeviceArray(dtype=np.uint64, count=n)
    maximum, unsorted = C.c_uint64(), C.c_int(-1)
    _check(call(_ctx(), C.byref(g.view), C.c_void_p(bounds.ptr), C.byref(maximum), C.byref(unsorted)))
    sums = [int(ew[indptr[v]:indptr[v + 1]].sum()) for v in range(n)]
    assert unsorted.value == (kind != "sorted")
    assert maximum.value == max(sums) and np.array_equal(bounds.get(), sums)


@pytest.mark.parametrize("name", list(GRAPHS))
@pytest.mark.parametrize("width", ["standard", "big"])
def test_parallel_entries_are_summed(hx, oracle, name, width):
    print(f"case parallel entries graph={name} width={width}", flush=True)
    c = GRAPHS[name]()
    g = hx.Graph(c["indptr"], c["indices"], width, c["edge_weights"], c["vertex_weights"])
    og = oracle.Graph(c["indptr"], c["indices"].astype(np.int32), c["edge_weights"], c["vertex_weights"])
    gh, oh = g.coarsen(4, 0, 1.0, 24, cluster_size_factor=16), oracle.coarsen(og, 4, 0, 1.0, 24, 16)
    assert len(gh) == len(oh) > 1
    for i in range(len(gh)):
        for x, y in zip(gh.level(i), oh.level(i).arrays()):
            assert np.array_equal(x, y), i
        if i + 1 < len(gh):
            assert np.array_equal(gh.map(i), oh.map(i)), i
    labels, rep = g.partition(2, 1.1, 0)
    expect, res = oracle.partition(og, 2, 1.1, 0)
    assert np.array_equal(labels, expect) and rep["final_cut"] == res.final_cut
