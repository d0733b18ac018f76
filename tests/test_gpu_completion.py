"""GPU: entry points that return host values synchronise the stream (gpart_hip.h): what they
write on the device is complete when they return, for readers on other streams too, also
where the kernel that writes it sends the host values itself."""
from __future__ import annotations

import ctypes as C

import pytest

from test_gpu_refine_rows import random_graph
from test_gpu_refine_rows_handle import Level, shuffled

pytestmark = pytest.mark.gpu

N, K = 20_001, 8


@pytest.mark.parametrize("form", ["cache", "rows"])
def test_arrays_are_complete_on_return(hx, form):
    if hx.device_count() < 1:
        pytest.skip("no GPU")
    print(f"case completion form={form}", flush=True)
    level = Level(hx, random_graph(hx, N, 26), K, form == "rows")
    D, ctx = level.D, level.D._ctx()
    level.L.gpart_ctx_stream.restype = C.c_void_p
    level.L.gpart_ctx_stream.argtypes = level.L.hipStreamQuery.argtypes = [C.c_void_p]
    stream = level.L.gpart_ctx_stream(ctx)

    def idle():
        return level.L.hipStreamQuery(stream) == 0

    for attempt in range(20):
        D._check(level.L.gpart_degree_classes_build(ctx, level.view(), level.classes()))
        assert idle(), ("classes", attempt)
        level.set_labels(shuffled(N, K, attempt))
        for step in (level.lp, lambda: level.rebalance(N // K)):
            rc, st = step()
            assert rc == 0 and st.movers > 0
            assert idle(), (step, attempt)
