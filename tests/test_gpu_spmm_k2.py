"""GPU test: two right-hand sides take no longer than four (27-point grid of 54^3, FP32: 9.7 and 11.2 us; with the entries of
a row fetched anew by every load 16.8 and 12.8)."""
import time

import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu


def test_two_columns_are_no_slower_than_four(gpu):
    m, n, cp, ri, val = fl.gen_matrix(fl.GEN_STENCIL27, 1, 0, 0, (54,))
    M = fl.FastLoadMatrix(m, n, cp, ri, val, width=64)
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
    assert best[2] < 1.08 * best[4]  # the middle of 0.87 and 1.31
