"""GPU test of Y = A X with more row lanes than one launch can have (2^32): 2^26 + 77 rows, k = 64 and X and Y at an odd
4-byte address, so that 64 lanes own a row. Rows on both sides of where the launches part, whole numbers."""
import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu


def test_more_rows_than_a_launch(gpu):
    m, n, k, cut = (1 << 26) + 77, 5, 64, 1 << 25
    full = np.array([0, 1, cut - 1, cut, cut + 3, 2 * cut - 1, 2 * cut, m - 1])
    rows, cols = np.repeat(full, n), np.tile(np.arange(n), full.size)
    vals = np.arange(1.0, rows.size + 1)
    o = np.lexsort((rows, cols))
    cp = np.concatenate([[0], np.cumsum(np.bincount(cols, minlength=n))]).astype(np.int32)
    M = fl.FastLoadMatrix(m, n, cp, rows[o].astype(np.int32), vals[o], width=64)
    M.prepare_rows()
    X = np.random.default_rng(0).integers(-3, 4, (n, k)).astype(np.float32)
    dX, dY = DeviceArray(n * k + 1, np.float32), DeviceArray(m * k + 1, np.float32)
    dX.view(1, n * k).copy_from(DeviceArray.from_host(X))
    seven = DeviceArray.from_host(np.full(k, 7, np.float32))
    seen = np.unique(np.clip(np.concatenate([full - 1, full, full + 1]), 0, m - 1))  # and the empty rows next to them
    for accumulate in (False, True):
        for r in seen:
            dY.view(1 + int(r) * k, k).copy_from(seven)
        M.spmm(dX.view(1, n * k), dY.view(1, m * k), k, fl.VAL_F32, accumulate=accumulate)
        for r in seen:
            mine = rows == r
            want = vals[mine].astype(np.float32) @ X[cols[mine]] + (7 if accumulate else 0)
            assert np.array_equal(dY.view(1 + int(r) * k, k).to_host(), want), r
