"""GPU test: two right-hand sides take no longer than four (27-point grid of 72^3, FP32: 19.6 and 20.2 us; with the entries of
a row fetched anew by every load 34.4 and 22.2)."""
import time

import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu


def test_two_columns_are_no_slower_than_four(gpu):
    m, n, cp, ri, val = fl.gen_matrix(fl.GEN_STENCIL27, 1, 0, 0, (72,))
    M = fl.FastLoadMatrix(m, n, cp, ri, val, width=64)
    M.prepare_rows()
    best = {2: np.inf, 4: np.inf}
    for _ in range(8):
        for k in best:
            X, Y = DeviceArray.zeros(n * k, np.float32), DeviceArray.zeros(m * k, np.float32)
            M.spmm(X, Y, k, fl.VAL_F32)
            fl.synchronize()
            t = time.perf_counter()
            for _ in range(200):
                M.spmm(X, Y, k, fl.VAL_F32)
            fl.synchronize()
            best[k] = min(best[k], time.perf_counter() - t)
    assert best[2] < 1.23 * best[4]  # the middle of 0.97 and 1.55
