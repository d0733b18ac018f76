"""Reductions that fold and publish themselves (hip/reduce.hpp): the weight statistics of a
graph at the edges of a thread's four loads, of one workgroup and of the largest grid, in
both widths, against numpy; sums that saturate (src/initial_partition_gpu.cu:31-35,
src/refine.cu:367-372)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIMIT = (2**63 - 1) // 2


@pytest.mark.parametrize("n", [1, 255, 257, 1023, 1024, 1025, 2049, 100_003, 2_097_152, 2_097_153])
@pytest.mark.parametrize("width", ["standard", "big"])
def test_weight_statistics(hx, n, width):
    from horkxg_amd.device import CsrView, DeviceArray, WIDTHS, _check, _ctx, hip_lib

    lib = hip_lib()
    for call, outputs in ((lib.gpart_vertex_weight_stats, 3), (lib.gpart_edge_weight_sum, 2),
                          (lib.gpart_max_edge_weight, 1)):
        call.argtypes = [C.c_void_p] * (2 + outputs)
    print(f"case reduce n={n} width={width}", flush=True)
    rng = np.random.default_rng(n)
    w_t = np.uint32 if width == "standard" else np.uint64
    inputs = [rng.integers(1, 2**32, n).astype(w_t)]
    if width == "big":
        inputs += [rng.integers(2**62, 2**64, n, dtype=np.uint64), np.full(n, LIMIT // n, np.uint64)]
    for w in inputs:
        d = DeviceArray(w, w_t)
        view = CsrView(n, n, WIDTHS[width], None, None, d.ptr, d.ptr)
        exact = sum(int(x) for x in np.add.reduceat(w.astype(object), range(0, n, 1 << 16))) if n > 1 else int(w[0])
        for _ in range(2):  # the second call finds the first one's counter cleared
            a, b, c = C.c_uint64(), C.c_uint64(), C.c_uint64()
            _check(lib.gpart_vertex_weight_stats(_ctx(), C.byref(view), C.byref(a), C.byref(b), C.byref(c)))
            assert (a.value, b.value, c.value) == (min(exact, 2**64 - 1), int(w.max()), int(w.min()))
            _check(lib.gpart_edge_weight_sum(_ctx(), C.byref(view), C.byref(a), C.byref(b)))
            assert (a.value, b.value) == (min(exact, 2**64 - 1), min(exact, LIMIT + 1))
            _check(lib.gpart_max_edge_weight(_ctx(), C.byref(view), C.byref(c)))
            assert c.value == int(w.max())
