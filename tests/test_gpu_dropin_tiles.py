"""GPU test of the line between the two ways of the drop-in y = A x: numbers of tiles and of repeated rows on both sides of
it, with tiles of one entry, full tiles, and columns of equal rows; y = A x takes both ways to the bound of the sum
of a row's products, and about as long as y += A x where the tiles are many and narrow."""
import time

import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray, KERNEL_DROPIN, VAL_F32, VAL_F64

pytestmark = pytest.mark.gpu


def _device(m, n, rows, cols, kind, width, rng):
    o = np.lexsort((rows, cols))
    rows, cols = rows[o], cols[o]
    dt = np.float64 if kind == VAL_F64 else np.float32
    val, x = rng.standard_normal(rows.size).astype(dt), rng.standard_normal(n).astype(dt)
    cp = np.concatenate([[0], np.cumsum(np.bincount(cols, minlength=n))]).astype(np.int32)
    M = fl.FastLoadMatrix(m, n, cp, rows.astype(np.int32), val.astype(np.float64), width=width)
    M.prepare(kind)
    dsx = DeviceArray.zeros(n, dt)
    M.permute_x(DeviceArray.from_host(x), dsx)
    prod = val.astype(np.float64) * x[cols].astype(np.float64)
    bound = (np.bincount(rows, minlength=m) + 2) * np.finfo(dt).eps * np.bincount(rows, np.abs(prod), m)
    return M, dsx, np.bincount(rows, prod, m), bound, dt


@pytest.mark.parametrize("width", [32, 64])
@pytest.mark.parametrize("kind", [VAL_F64, VAL_F32], ids=["f64", "f32"])
@pytest.mark.parametrize("shape", ["narrow", "full", "dense"])
def test_both_sides(gpu, width, kind, shape):
    rng = np.random.default_rng(1)
    tiles = (132 if kind == VAL_F64 else 192) * 64 // width  # the most that take one launch
    for t in (1, tiles - 1, tiles, tiles + 1):
        if shape == "narrow":  # a tile for every entry of one column
            m, n, rows, cols = 8000, 1, rng.choice(8000, t, replace=False), np.zeros(t, int)
        elif shape == "full":  # `width` columns of t entries, no row twice in a tile
            m, n = 8192, width
            rows, cols = (np.arange(t)[:, None] + 401 * np.arange(width)[None, :]).ravel() % m, np.tile(np.arange(width), t)
        else:  # full columns: every tile is one row
            m = n = max(1, int((t * width) ** 0.5))
            rows, cols = np.tile(np.arange(m), n), np.repeat(np.arange(n), m)
        M, dsx, ref, bound, dt = _device(m, n, rows, cols, kind, width, rng)
        dy = DeviceArray.from_host(np.full(m, 7, dt))
        M.spmv(dsx, dy, KERNEL_DROPIN, kind, assign=True)
        assert np.all(np.abs(dy.to_host() - ref) <= bound), (t, M.tilenum)


@pytest.mark.parametrize("kind", [VAL_F64, VAL_F32], ids=["f64", "f32"])
def test_many_narrow_tiles(gpu, kind):
    """A column of 5,000 entries: 6.5 us in a stream of calls, 79 to 117 in one workgroup."""
    rng = np.random.default_rng(2)
    M, dsx, _, _, dt = _device(8000, 1, rng.choice(8000, 5000, replace=False), np.zeros(5000, int), kind, 64, rng)
    dy = DeviceArray.zeros(8000, dt)

    def took(assign):
        best = np.inf
        for _ in range(5):
            fl.synchronize()
            t = time.perf_counter()
            for _ in range(500):
                M.spmv(dsx, dy, KERNEL_DROPIN, kind, assign=assign)
            fl.synchronize()
            best = min(best, time.perf_counter() - t)
        return best

    took(False)
    assert took(True) < 4 * took(False)
