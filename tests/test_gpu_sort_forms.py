"""The stable sort operator at the limits of its forms: one, two and three
radix passes, blocks of 4096 and 8192 keys, ragged ends, crowded and empty
stretches of cells (GPU)."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import _gpu_sort

pytestmark = pytest.mark.gpu


# one pass up to 1023 cells, two from 1024, three from 2^20; blocks of 8192 keys where the table of the
# smaller ones does not fit (40000 keys of 700 cells, 2^22 of 2^18)
@pytest.mark.parametrize("n,cells", [(1, 1), (4095, 1), (4097, 1023), (4096, 1024), (40000, 700), (8193, 1025),
                                     (100000, (1 << 20) - 1), (5000, 1 << 20), (3000, 1 << 24),
                                     ((1 << 21) + 1, 40000), ((1 << 22) + 5, 1 << 18)])
@pytest.mark.parametrize("crowd", [0.0, 0.7])
def test_sort_forms(n, cells, crowd):
    print(f"sort n={n} cells={cells} crowd={crowd}", flush=True)
    rng = np.random.default_rng(n + cells)
    keys = rng.integers(0, cells, n).astype(np.uint32)
    keys[rng.random(n) < crowd] = cells // 2
    keys[rng.random(n) < 0.02] = rng.choice([cells, cells + 7, 0xFFFFFFFF])
    perm, start = _gpu_sort(keys, cells)
    order = np.argsort(np.minimum(keys, cells), kind="stable")
    want = np.searchsorted(np.minimum(keys, cells)[order], np.arange(cells + 1))
    assert np.array_equal(start, want)
    assert np.array_equal(perm, order[: want[-1]])
