"""Sorts of at most 8192 keys in one launch (hip/primitives.hip, rank_sort_kernel): every
entry's place is counted against all keys. Sizes at the edges of a run of 64 keys, of a
workgroup's 16 entries and of the form itself; 32- and 64-bit digits; ties with the largest
digit, which the lanes past the end hold too."""
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
