"""GPU test of the row pointers of the row order and of the heavy part of HYB where rows without entries come in
long runs: at the start, in the middle, at the end, and m much larger than the number of entries. Values and
x are small whole numbers, so every y is exact."""
import time

import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu


def _matrix(m, n, rows):
    """A column for each row in turn; several entries may share a position."""
    cols = np.arange(rows.size) % n
    o = np.lexsort((rows, cols))
    cp = np.concatenate([[0], np.cumsum(np.bincount(cols, minlength=n))]).astype(np.int32)
    return cols, o, cp


@pytest.mark.parametrize("m", [1, 255, 256, 511, 512, 513, 70_000, 300_001])
@pytest.mark.parametrize("where", ["one", "first", "last", "ends", "middle", "few"])
def test_runs_of_empty_rows(gpu, m, where):
    rng = np.random.default_rng(m)
    n = 37
    rows = {"one": np.array([m - 1]), "first": rng.integers(0, max(m // 9, 1), 5000),
            "last": m - 1 - rng.integers(0, max(m // 9, 1), 5000), "ends": np.repeat([0, m - 1], [7, 4000]),
            "middle": np.full(513, m // 2), "few": rng.integers(0, m, 9)}[where]
    cols, o, cp = _matrix(m, n, rows)
    vals = rng.integers(1, 4, rows.size).astype(float)
    x = rng.integers(-3, 4, n).astype(np.float32)
    M = fl.FastLoadMatrix(m, n, cp, rows[o].astype(np.int32), vals[o], width=64)
    want = np.bincount(rows, vals * x[cols], m).astype(np.float32)
    dx, dsx, dy = DeviceArray.from_host(x), DeviceArray(n, np.float32), DeviceArray.from_host(np.full(m, 7, np.float32))
    M.prepare_rows()
    M.spmm(dx, dy, 1, fl.VAL_F32)
    assert np.array_equal(dy.to_host(), want)
    M.prepare(fl.VAL_F32)
    M.prepare_hyb(n, 128, 1024)
    M.permute_x(dx, dsx)
    M.spmv(dsx, dy, fl.KERNEL_HYB, fl.VAL_F32, assign=True)
    assert np.array_equal(dy.to_host(), want)


def test_long_run_is_not_written_by_one_lane(gpu):
    """8 M rows, entries in the first 100 K: 1.5 ms, and 200 ms where one lane writes the empty rows' pointers."""
    m, n = 8_000_000, 100_000
    rows = np.random.default_rng(1).integers(0, 100_000, 1_000_000)
    cols, o, cp = _matrix(m, n, rows)
    best = np.inf
    for _ in range(3):
        M = fl.FastLoadMatrix(m, n, cp, rows[o].astype(np.int32), np.ones(rows.size), width=64)
        t = time.perf_counter()
        M.prepare_rows()
        best = min(best, time.perf_counter() - t)
        M.close()
    assert best < 0.05
