"""GPU test: two right-hand sides take about as long as four (100 K uniform rows of 32 entries, FP32: 19 us each); with the
entries of a row fetched anew by every load they took 28 against 20."""
import time

import numpy as np

import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu


def test_two_columns_are_no_slower_than_four(gpu):
    m = n = 100_000
    rng = np.random.default_rng(0)
    rows, cols = np.repeat(np.arange(m), 32), rng.integers(0, n, 32 * m)
    o = np.lexsort((rows, cols))
    cp = np.concatenate([[0], np.cumsum(np.bincount(cols, minlength=n))]).astype(np.int32)
    M = fl.FastLoadMatrix(m, n, cp, rows[o].astype(np.int32), np.ones(rows.size), width=64)
    M.prepare_rows()
    best = {2: np.inf, 4: np.inf}
    for _ in range(8):
        for k in best:
            X, Y = DeviceArray.zeros(n * k, np.float32), DeviceArray.zeros(m * k, np.float32)
            M.spmm(X, Y, k, fl.VAL_F32)
            fl.synchronize()
            t = time.perf_counter()
            for _ in range(300):
                M.spmm(X, Y, k, fl.VAL_F32)
            fl.synchronize()
            best[k] = min(best[k], time.perf_counter() - t)
    assert best[2] < 1.2 * best[4]
