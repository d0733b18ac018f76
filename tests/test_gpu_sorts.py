"""Sorts (hip/primitives.hip) at the edges of their forms: the passes' tiles of 2048 keys below
2^21 keys and of 4096 keys from there on, and sorts of at most 8192 keys in one launch (rank_sort_kernel),
where every entry's place is counted against all keys: sizes at the edges of a run of 64
keys, of a workgroup's 16 entries and of the form itself; 32- and 64-bit digits; ties with
the largest digit, which the lanes past the end hold too."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 15, 16, 17, 63, 64, 65, 1023, 1025, 8191, 8192])
@pytest.mark.parametrize("bits", [(0, 32), (0, 33), (0, 64), (40, 64)])
def test_rank_sort(hx, n, bits):
    begin, end = bits
    print(f"case rank sort n={n} bits={bits}", flush=True)
    rng = np.random.default_rng(n)
    mask = np.uint64(2**64 - 1 if end - begin == 64 else (1 << (end - begin)) - 1)
    largest = rng.integers(0, 2**64, n, dtype=np.uint64) | (mask << np.uint64(begin))
    few = rng.integers(0, 3, n).astype(np.uint64) << np.uint64(begin)
    for keys in (largest, few, np.where(rng.random(n) < 0.5, largest, few)):
        order = np.argsort((keys >> np.uint64(begin)) & mask, kind="stable")
        vals = np.arange(n, dtype=np.uint32)
        k, v = hx.device.sort_pairs(keys, vals, begin, end)
        assert np.array_equal(v, vals[order])
        assert np.array_equal(k, keys[order])


@pytest.mark.parametrize("n", [2**21 - 1, 2**21, 2**21 + 1, 2**21 + 4097])
def test_large_tiles(hx, n):
    print(f"case sort passes n={n}", flush=True)
    rng = np.random.default_rng(n)
    keys = rng.integers(0, 2**64, n, dtype=np.uint64)
    keys[: n // 2] &= np.uint64(~(0x3FFF << 5) & (2**64 - 1))  # half the keys share a digit
    order = np.argsort((keys >> np.uint64(5)) & np.uint64(0x3FFF), kind="stable")
    vals = np.arange(n, dtype=np.uint32)
    k, v = hx.device.sort_pairs(keys, vals, 5, 19)
    assert np.array_equal(v, vals[order])
    assert np.array_equal(k, keys[order])
    vals64 = keys ^ np.uint64(7)
    assert np.array_equal(hx.device.sort_pairs(keys, vals64, 5, 19)[1], vals64[order])
    assert np.array_equal(hx.device.sort_pairs(keys, None, 5, 19), keys[order])
