"""GPU test of the drop-in y = A x of small matrices (one workgroup, y in LDS): sizes on both sides of
its limits (8,192 rows; 8,192 FP64 or 12,288 FP32 entries), both tile widths, empty rows and columns, a
full row, and y's old contents. Against FP64 on the host: each product and sum rounds once, so a
row of c entries is within (c + 2) eps of the sum of its products' magnitudes."""
import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray, KERNEL_DROPIN, VAL_F32, VAL_F64

pytestmark = pytest.mark.gpu


def _matrix(m, n, nnz, rng):
    """nnz distinct positions: one full row if it fits, the rest anywhere; some rows and columns stay empty."""
    flat = rng.choice(m * n, nnz, replace=False) if m * n > nnz else np.arange(m * n)
    if m > 1 and nnz >= 2 * n:
        full = (m // 2) * n + np.arange(n)
        flat = np.concatenate([full, np.setdiff1d(flat, full)])[:nnz]
    col, row = np.divmod(np.sort((flat % n) * m + flat // n), m)
    cp = np.concatenate([[0], np.cumsum(np.bincount(col, minlength=n))]).astype(np.int32)
    return cp, row.astype(np.int32), col


@pytest.mark.parametrize("m,n,nnz", [(1, 1, 1), (1, 5000, 5000), (5000, 1, 5000), (63, 65, 129), (1138, 1138, 4094),
                                     (8192, 300, 8192), (8193, 300, 8192), (300, 700, 8193), (2000, 2000, 12288),
                                     (2000, 2000, 12289), (100, 64, 6400)])
@pytest.mark.parametrize("width", [32, 64])
@pytest.mark.parametrize("kind", [VAL_F64, VAL_F32])
def test_small_assign(gpu, m, n, nnz, width, kind):
    rng = np.random.default_rng(m + 3 * n + nnz)
    cp, ri, col = _matrix(m, n, nnz, rng)
    dt = np.float64 if kind == VAL_F64 else np.float32
    val = rng.standard_normal(len(ri)).astype(dt)
    x = rng.standard_normal(n).astype(dt)
    M = fl.FastLoadMatrix(m, n, cp, ri, val.astype(np.float64), width=width)
    M.prepare(kind)
    dsx = DeviceArray.zeros(n, dt)
    M.permute_x(DeviceArray.from_host(x), dsx)
    prod = val.astype(np.float64) * x[col].astype(np.float64)
    ref, mag = np.bincount(ri, prod, m), np.bincount(ri, np.abs(prod), m)
    bound = (np.bincount(ri, minlength=m) + 2) * np.finfo(dt).eps * mag
    dy = DeviceArray.from_host(np.full(m, 7, dt))
    for _ in range(2):
        M.spmv(dsx, dy, KERNEL_DROPIN, kind, assign=True)
        assert np.all(np.abs(dy.to_host() - ref) <= bound)
    y = np.arange(m).astype(dt)
    dy = DeviceArray.from_host(y)
    M.spmv(dsx, dy, KERNEL_DROPIN, kind)  # y += A x
    assert np.all(np.abs(dy.to_host() - (ref + y)) <= bound + (np.bincount(ri, minlength=m) + 2) * np.finfo(dt).eps * y)


@pytest.mark.parametrize("kind", [VAL_F64, VAL_F32])
def test_small_assign_nonfinite(gpu, kind):
    dt = np.float64 if kind == VAL_F64 else np.float32
    cp, ri, col = _matrix(70, 90, 400, np.random.default_rng(5))
    val = np.ones(len(ri))
    x = np.ones(90, dt)
    x[3], x[40] = np.inf, np.nan
    M = fl.FastLoadMatrix(70, 90, cp, ri, val, width=64)
    M.prepare(kind)
    dsx = DeviceArray.zeros(90, dt)
    M.permute_x(DeviceArray.from_host(x), dsx)
    dy = DeviceArray.from_host(np.full(70, np.nan, dt))
    M.spmv(dsx, dy, KERNEL_DROPIN, kind, assign=True)
    assert np.array_equal(dy.to_host(), np.bincount(ri, val * x[col], 70).astype(dt), equal_nan=True)
