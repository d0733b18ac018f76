"""GPU: the handle of the refinement rounds without a cache (gpart_refine_rows_*), called
round by round as the C ABI allows: labels that the caller changes between two rounds, and
rounds of another level or part count, beside the cached rounds
(src/refine_incremental.cuh:235-361). Everything is whole numbers and must be equal."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from test_gpu_refine_rows import hub_graph, random_graph

pytestmark = pytest.mark.gpu

INVALID_ARGUMENT = 1


class Status(C.Structure):
    _fields_ = [("movers", C.c_int64), ("cut_delta", C.c_int64), ("candidates", C.c_int64),
                ("max_part_weight", C.c_uint64), ("part_weights", C.c_uint64 * 32), ("mover_entries", C.c_int64),
                ("rebuilt", C.c_int32), ("cut_after", C.c_uint64)]

    def values(self, k):
        return (self.movers, self.cut_delta, self.candidates, self.max_part_weight, list(self.part_weights[:k]),
                self.mover_entries)


class Level:
    """A level's arrays as a caller of the rounds keeps them; rows: its handle, or cached rounds."""

    def __init__(self, hx, csr, k, rows):
        from horkxg_amd import device as D

        self.D, self.k, self.L = D, k, D.hip_lib()
        vp, i32, u64 = C.c_void_p, C.c_int, C.c_uint64
        bind = {
            "gpart_part_weights": [vp, vp, vp, i32, vp],
            "gpart_refine_build_cache": [vp, vp, vp, vp, i32, vp, i32],
            "gpart_refine_lp_round": [vp, vp, vp, vp, i32, vp, i32, C.c_double, vp, vp, vp, vp, vp, vp],
            "gpart_refine_rebalance_round": [vp, vp, vp, vp, i32, vp, i32, vp, u64, vp, vp, vp],
            "gpart_refine_rows_create": [vp, vp, vp, i32, i32, vp],
            "gpart_refine_rows_destroy": [vp],
            "gpart_refine_rows_reset": [vp],
            "gpart_refine_rows_check": [vp, vp, vp, vp, vp, vp, i32, vp, u64, vp, vp],
            "gpart_refine_lp_round_rows": [vp, vp, vp, vp, vp, vp, i32, C.c_double, vp, vp, vp, vp, vp, vp],
            "gpart_refine_rebalance_round_rows": [vp, vp, vp, vp, vp, vp, i32, vp, u64, vp, vp, vp],
        }
        for name, types in bind.items():
            getattr(self.L, name).argtypes = types
        self.g = g = D.DeviceGraph(*csr)
        n = g.n
        self.cache = D.DeviceArray(dtype=np.uint32, count=n * k)
        self.targets = D.DeviceArray(dtype=np.int32, count=n)
        self.gains = D.DeviceArray(dtype=np.int64, count=n)
        self.flags = D.DeviceArray(np.zeros(n), np.int32)
        self.weights = D.DeviceArray(dtype=np.uint64, count=k)
        self.rows = C.c_void_p()
        self.with_rows = rows
        if rows:
            D._check(self.L.gpart_refine_rows_create(D._ctx(), self.view(), self.classes(), k, 4, C.byref(self.rows)))
            assert self.rows.value

    def __del__(self):
        if self.rows:
            self.L.gpart_refine_rows_destroy(self.rows)

    def view(self):
        return C.byref(self.g.view)

    def classes(self):
        return C.byref(self.g.classes)

    def set_labels(self, labels):
        """Other labels in the place of the ones the rounds have led to."""
        D, ctx = self.D, self.D._ctx()
        self.labels, self.locks = D.DeviceArray(labels, np.int32), D.DeviceArray(np.zeros(self.g.n), np.int32)
        D._check(self.L.gpart_part_weights(ctx, self.view(), self.labels.ptr, self.k, self.weights.ptr))
        if self.with_rows:
            D._check(self.L.gpart_refine_rows_reset(self.rows))
        else:
            D._check(self.L.gpart_refine_build_cache(ctx, self.view(), self.classes(), self.labels.ptr, self.k,
                                                     self.cache.ptr, 4))

    def lp(self, k=None):
        st, k = Status(), k or self.k
        tail = (self.labels.ptr, k, 0.25, self.locks.ptr, self.targets.ptr, self.gains.ptr, self.flags.ptr,
                self.weights.ptr, C.byref(st))
        head = (self.D._ctx(), self.view(), self.classes())
        if self.with_rows:
            return self.L.gpart_refine_lp_round_rows(*head, self.rows, self.cache.ptr, *tail), st
        return self.L.gpart_refine_lp_round(*head, self.cache.ptr, 4, *tail), st

    def rebalance(self, capacity, k=None):
        st, k = Status(), k or self.k
        tail = (self.labels.ptr, k, self.weights.ptr, capacity, self.targets.ptr, self.flags.ptr, C.byref(st))
        head = (self.D._ctx(), self.view(), self.classes())
        if self.with_rows:
            return self.L.gpart_refine_rebalance_round_rows(*head, self.rows, self.cache.ptr, *tail), st
        return self.L.gpart_refine_rebalance_round(*head, self.cache.ptr, 4, *tail), st

    def differing(self, capacity=None):
        """Entries of the rows the next round sums that differ from a build from the labels."""
        D, out = self.D, C.c_int64(-1)
        expected = D.DeviceArray(dtype=np.uint32, count=self.g.n * self.k)
        head = (D._ctx(), self.view(), self.classes())
        D._check(self.L.gpart_refine_build_cache(*head, self.labels.ptr, self.k, expected.ptr, 4))
        D._check(self.L.gpart_refine_rows_check(*head, self.rows, self.cache.ptr, self.labels.ptr, self.k,
                                                None if capacity is None else self.weights.ptr, capacity or 0,
                                                expected.ptr, C.byref(out)))
        return out.value


@pytest.fixture(scope="module", autouse=True)
def need_gpu(hx):
    if hx.device_count() < 1:
        pytest.skip("no GPU")


def shuffled(n, k, seed):
    return (np.random.default_rng(seed).permutation(n) % k).astype(np.int32)


@pytest.mark.parametrize("name,k", [("hubs", 8), ("hubs", 32), ("random", 5)])
def test_labels_changed_between_rounds(hx, name, k):
    print(f"case rows handle labels graph={name} k={k}", flush=True)
    csr = hub_graph(hx, 12_001, 24) if name == "hubs" else random_graph(hx, 20_001, 26)
    n = len(csr[0]) - 1
    cached, rows = Level(hx, csr, k, False), Level(hx, csr, k, True)
    for seed in (1, 2):  # the second labels take the place of those the first rounds led to
        for level in (cached, rows):
            level.set_labels(shuffled(n, k, seed))
        for step in range(4):
            results = []
            for level in (cached, rows):
                rc, st = level.lp() if step % 2 == 0 else level.rebalance(n // k)
                assert rc == 0
                results.append((st.values(k), level.labels.get()))
            assert results[0][0] == results[1][0], (seed, step)
            assert np.array_equal(results[0][1], results[1][1]), (seed, step)
            assert results[0][0][0] > 0


def test_rounds_of_another_level_are_refused(hx):
    print("case rows handle refusals", flush=True)
    csr, other = hub_graph(hx, 12_001, 24), random_graph(hx, 20_001, 26)
    level = Level(hx, csr, 8, True)
    level.set_labels(shuffled(12_001, 8, 1))
    before = level.labels.get()
    for k in (1, 7, 9, 32, 33):
        assert level.lp(k)[0] == INVALID_ARGUMENT and level.rebalance(1600, k)[0] == INVALID_ARGUMENT
    level.g, mine = level.D.DeviceGraph(*other), level.g
    assert level.lp()[0] == INVALID_ARGUMENT and level.rebalance(1600)[0] == INVALID_ARGUMENT
    level.g = mine
    assert level.L.gpart_refine_rows_reset(None) == INVALID_ARGUMENT
    assert np.array_equal(level.labels.get(), before)
    rc, st = level.lp()  # a refused round leaves the handle as it was
    assert rc == 0 and st.movers > 0


@pytest.mark.parametrize("name,k", [("hubs", 8), ("hubs", 31), ("random", 5)])
def test_check_finds_rows_of_other_labels(hx, name, k):
    """What the strict checks compare: nothing differs before and after rounds, and rows
    summed from other labels than the ones given are found."""
    print(f"case rows check graph={name} k={k}", flush=True)
    csr = hub_graph(hx, 12_001, 24) if name == "hubs" else random_graph(hx, 20_001, 26)
    n = len(csr[0]) - 1
    level = Level(hx, csr, k, True)
    level.set_labels(shuffled(n, k, 1))
    for step in range(4):
        assert level.differing() == 0 and level.differing(n // k) == 0, step
        rc, st = level.lp() if step % 2 == 0 else level.rebalance(n // k)
        assert rc == 0 and st.movers > 0
    assert level.differing() == 0
    other = level.labels.get()
    v = int(csr[1][csr[0][n // 2]])  # of some row: its neighbours' rows change
    other[v] = (other[v] + 1) % k
    level.D._check(level.L.gpart_memcpy_htod(level.D._ctx(), C.c_void_p(level.labels.ptr), other.ctypes.data, 4 * n))
    assert level.differing() == 2 * (csr[0][v + 1] - csr[0][v])  # each neighbour: an entry less, an entry more
    level.L.gpart_refine_rows_reset(level.rows)
    assert level.differing() == 0


def test_strict_verification_checks_the_rows(hx):
    """verify=True builds a cache and sums the rows once more for every round."""
    print("case rows strict", flush=True)
    indptr, indices = random_graph(hx, 20_001, 26)
    g = hx.Graph(indptr, indices)
    start = shuffled(20_001, 8, 1)
    launches = []
    for verify in (False, True):
        hx.profile_reset()
        hx.profile_enable("refine_cache", True)
        try:
            labels, rep = g.refine(start, 8, 1.03, 6, 3, verify=verify)
            launches.append(hx.profile_read("refine_cache")["launches"])
        finally:
            hx.profile_enable("refine_cache", False)
    rounds = rep["rounds"] + rep["admission_iterations"]
    assert rep["admission_iterations"] > 0
    assert launches == [rounds, 3 * rounds]
