"""GPU test of the preparation's scans and sorts at the sizes where their launches change: scans around one
tile (2,048), one workgroup (16,384) and 4,096 tiles; radix sorts of one to four passes, around one tile of 4,096
keys. Whole-number data, so every product is exact."""
import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu


def _csc(m, n, lengths, rng):
    cp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    first = rng.integers(0, m, n)
    step = m // max(int(lengths.max()), 1)  # distinct rows, ascending after the sort below
    col = np.repeat(np.arange(n), lengths)
    row = (first[col] + (np.arange(len(col)) - cp[col]) * max(step, 1)) % m
    order = np.lexsort((row, col))
    return cp, row[order].astype(np.int32), col


@pytest.mark.parametrize("n", [1, 2047, 2049, 4096, 16383, 16384, 16385, 70001, 8388608, 8390657])
def test_columns(gpu, n):
    """The column sort (scan of n level flags) and the layout that follows from it."""
    rng = np.random.default_rng(n)
    m = 16
    lengths = rng.integers(0, 2 if n > 1 << 20 else 5, n)
    cp, ri, col = _csc(m, n, lengths, rng)
    val = rng.integers(-4, 5, len(ri)).astype(np.float64)
    x = rng.integers(-4, 5, n).astype(np.float64)
    M = fl.FastLoadMatrix(m, n, cp, ri, val, width=64)
    assert np.array_equal(M.perm(), np.argsort(lengths, kind="stable"))
    M.prepare_rows()
    dy = DeviceArray.zeros(m, np.float64)
    M.spmm(DeviceArray.from_host(x), dy, 1, fl.VAL_F64)
    assert np.array_equal(dy.to_host(), np.bincount(ri, val * x[col], m))


@pytest.mark.parametrize("m", [2, 256, 257, 65536, 65537, 16777216, 16777217])
@pytest.mark.parametrize("n,per", [(40, 2), (500, 9), (40001, 9)])
def test_rows(gpu, m, n, per):
    """Sorts by row (one to four passes) of fewer and more entries than a sort tile, for every schedule."""
    rng = np.random.default_rng(m + n)
    lengths = rng.integers(0, min(per, m) + 1, n)
    cp, ri, col = _csc(m, n, lengths, rng)
    val = rng.integers(-4, 5, len(ri)).astype(np.float64)
    x = rng.integers(-4, 5, n).astype(np.float64)
    want = np.bincount(ri, val * x[col], m)
    M = fl.FastLoadMatrix(m, n, cp, ri, val, width=64)
    dx, dsx, dy = DeviceArray.from_host(x), DeviceArray.zeros(n, np.float64), DeviceArray.zeros(m, np.float64)
    M.prepare_rows()
    M.spmm(dx, dy, 1, fl.VAL_F64)
    assert np.array_equal(dy.to_host(), want)
    M.permute_x(dx, dsx)
    for kernel in (fl.KERNEL_WIN, fl.KERNEL_WINR, fl.KERNEL_PB, fl.KERNEL_HYB):
        if kernel == fl.KERNEL_HYB:
            M.prepare_hyb(min(n, 1000), 128, 16384)
        else:
            M.prepare_schedule(kernel, 64, 16384)
        M.spmv(dsx, dy, kernel, fl.VAL_F64, assign=True)
        assert np.array_equal(dy.to_host(), want), kernel
