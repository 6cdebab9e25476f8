"""GPU test of the radix sort (through csr_to_csc, a stable sort by column): one to four passes, key counts around
a wave, a tile (4,096) and the groups of eight tiles, all columns equal, ascending and random."""
import numpy as np
import pytest

import fastload_amd as fl

pytestmark = pytest.mark.gpu

SIZES = [(n, nnz) for n in (2, 256, 257, 65537) for nnz in (1, 63, 65, 1023, 1025, 4095, 4096, 4097, 32768, 36865, 300001)]
SIZES += [(16777217, nnz) for nnz in (1, 4097, 300001)]


@pytest.mark.parametrize("n,nnz", SIZES)
@pytest.mark.parametrize("order", ["random", "ascending", "equal"])
def test_stable_sort(gpu, n, nnz, order):
    rng = np.random.default_rng(n + nnz)
    col = rng.integers(0, n, nnz).astype(np.int32)
    if order == "ascending":
        col.sort()
    elif order == "equal":
        col[:] = n - 1
    m = 1 + nnz // 3
    rowptr = np.concatenate([[0], np.sort(rng.integers(0, nnz + 1, m - 1)), [nnz]]).astype(np.int32)
    val = rng.standard_normal(nnz)
    cval, crow, cptr, cnt, _ = fl.csr_to_csc(m, n, val, rowptr, col)
    o = np.argsort(col, kind="stable")
    assert np.array_equal(cval, val[o])
    assert np.array_equal(crow, np.repeat(np.arange(m), np.diff(rowptr))[o])
    assert np.array_equal(cnt, np.bincount(col, minlength=n))
    assert np.array_equal(cptr, np.concatenate([[0], np.cumsum(np.bincount(col, minlength=n))]))
