"""GPU test of the HYB schedule's row order (one workgroup per window): row counts around slices, rounds and
windows, rows with more than 255 heavy entries (a second pass) and windows without, all columns heavy and
some, FP32 values prepared before the schedule (written with it) and after. Whole-number data: exact."""
import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 63, 65, 1023, 1025, 4097, 16384, 16385, 40000])
@pytest.mark.parametrize("R", [1024, 16384])
@pytest.mark.parametrize("heavy", [600, 200])
@pytest.mark.parametrize("f32_first", [True, False])
def test_hyb_order(gpu, m, R, heavy, f32_first):
    rng = np.random.default_rng(m + R)
    n = 600
    density = np.minimum(rng.pareto(0.7, m) * 0.004, 1.0)  # rows of a few entries up to all 600
    density[m // 2] = 1.0
    B = rng.random((n, m)) < density  # by column
    ri = np.nonzero(B)[1].astype(np.int32)
    lengths = B.sum(1)
    cp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    val = rng.integers(-4, 5, len(ri)).astype(np.float64)
    x = rng.integers(-4, 5, n).astype(np.float64)
    want = np.bincount(ri, val * np.repeat(x, lengths), m)
    M = fl.FastLoadMatrix(m, n, cp, ri, val, width=64)
    if f32_first:
        M.prepare(fl.VAL_F32)
    M.prepare_hyb(heavy, 64, R)
    M.prepare(fl.VAL_F32)
    for kind, dt in ((fl.VAL_F64, np.float64), (fl.VAL_F32, np.float32)):
        dsx, dy = DeviceArray.zeros(n, dt), DeviceArray.from_host(np.full(m, 3, dt))
        M.permute_x(DeviceArray.from_host(x.astype(dt)), dsx)
        M.spmv(dsx, dy, fl.KERNEL_HYB, kind, assign=True)
        assert np.array_equal(dy.to_host(), want)
