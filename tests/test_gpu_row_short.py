"""GPU test of the row kernel for one vector on short rows (two lanes per row, up to six entries on average) against
the one for longer rows: a matrix alone and the same matrix above one of long rows give the same bits,
at row counts around a wave and a workgroup, with empty rows and rows of up to 40 entries."""
import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu


def _product(m, n, rows, cols, vals, x, y, kind, dt, accumulate):
    o = np.lexsort((rows, cols))
    cp = np.concatenate([[0], np.cumsum(np.bincount(cols, minlength=n))]).astype(np.int32)
    M = fl.FastLoadMatrix(m, n, cp, rows[o].astype(np.int32), vals[o], width=64)
    M.prepare_rows()
    dy = DeviceArray.from_host(y.astype(dt))
    M.spmm(DeviceArray.from_host(x.astype(dt)), dy, 1, kind, accumulate=accumulate)
    return dy.to_host()


@pytest.mark.parametrize("m", [1, 31, 32, 33, 127, 128, 129, 5003])
@pytest.mark.parametrize("kind,dt,tol", [(fl.VAL_F32, np.float32, 1e-5), (fl.VAL_F64, np.float64, 1e-12)],
                         ids=["f32", "f64"])
@pytest.mark.parametrize("accumulate", [False, True])
def test_short_rows(gpu, m, kind, dt, tol, accumulate):
    rng = np.random.default_rng(m)
    n, tall = 50, 4000
    lens = rng.integers(0, 6, m)
    lens[::9] = np.minimum(rng.integers(6, 41, lens[::9].size), 6 * m // max(1, lens[::9].size) if m < 9 else 40)
    while lens.sum() > 6 * m:
        lens[np.argmax(lens)] //= 2
    lens[0] = max(lens[0], 1)
    lens2 = rng.integers(30, 41, max(tall, m))  # the stacked matrix then has more than six per row
    rows = np.repeat(np.arange(m), lens)
    cols = np.concatenate([rng.choice(n, k, replace=False) for k in lens])
    vals = rng.standard_normal(rows.size).astype(np.float32).astype(np.float64)
    rows2 = np.repeat(np.arange(lens2.size), lens2) + m
    cols2 = np.concatenate([rng.choice(n, k, replace=False) for k in lens2]) + n
    x = rng.standard_normal(2 * n).astype(np.float32).astype(np.float64)
    y = rng.standard_normal(m + lens2.size).astype(np.float32).astype(np.float64)
    alone = _product(m, n, rows, cols, vals, x[:n], y[:m], kind, dt, accumulate)
    both = _product(m + lens2.size, 2 * n, np.r_[rows, rows2], np.r_[cols, cols2], np.r_[vals, np.ones(rows2.size)], x, y,
                    kind, dt, accumulate)
    want = np.bincount(rows, vals * x[cols], m) + (y[:m] if accumulate else 0)
    scale = np.bincount(rows, np.abs(vals * x[cols]), m) + (np.abs(y[:m]) if accumulate else 0)
    assert np.all(np.abs(alone - want) <= tol * scale)
    assert np.array_equal(alone, both[:m])
