"""GPU test of the PB and HYB schedules at the row counts where the band height chosen for the matrix
changes: 1,024 rows up to 262,144 rows, then the next multiple of 1,024 that keeps 256 bands, 16,384 rows
above 4.19 M rows; a last band of 1 to 3 rows; and a band height asked for that is no multiple of 64."""
import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu

TOL = {fl.VAL_F64: 1e-12, fl.VAL_F32: 1e-5}


@pytest.mark.parametrize("m", [1023, 1025, 262144, 262147, 700001, 4194305])
@pytest.mark.parametrize("kernel", [fl.KERNEL_PB, fl.KERNEL_HYB], ids=["pb", "hyb"])
@pytest.mark.parametrize("bt,R", [(64, 16384), (256, 16384), (128, 1500)])
def test_band_heights(gpu, m, kernel, bt, R):
    rng = np.random.default_rng(m)
    n = 3000
    lens = np.minimum(rng.zipf(1.7, n), 900)
    cols = np.repeat(np.arange(n), lens)
    rows = np.concatenate([np.sort(rng.choice(m, k, replace=False)) for k in lens])
    rows[np.cumsum(lens) - 1] = m - 1  # the last row gets an entry of every column
    vals = rng.standard_normal(rows.size).astype(np.float32).astype(np.float64)
    cp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    x = rng.standard_normal(n).astype(np.float32).astype(np.float64)
    want = np.bincount(rows, vals * x[cols], m)
    scale = np.bincount(rows, np.abs(vals * x[cols]), m)
    M = fl.FastLoadMatrix(m, n, cp, rows.astype(np.int32), vals, width=64)
    M.prepare(fl.VAL_F32)
    if kernel == fl.KERNEL_PB:
        M.prepare_schedule(kernel, bt, R)
    else:
        M.prepare_hyb(700, bt, R)
    for kind, dt in ((fl.VAL_F64, np.float64), (fl.VAL_F32, np.float32)):
        dsx, dy = DeviceArray(n, dt), DeviceArray.from_host(np.ones(m, dt))
        M.permute_x(DeviceArray.from_host(x.astype(dt)), dsx)
        M.spmv(dsx, dy, kernel, kind, assign=True)
        assert np.all(np.abs(dy.to_host() - want) <= TOL[kind] * scale)
        M.spmv(dsx, dy, kernel, kind)  # accumulate
        assert np.all(np.abs(dy.to_host() - 2 * want) <= 2 * TOL[kind] * scale)
