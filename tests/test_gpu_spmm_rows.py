"""GPU test of the row kernels at the edges of their steps: rows of 0 to 40 entries (a step is 16 entries;
with one right-hand side a lane loads four of them at a time, up to the arrays' end), row counts around a wave's and a workgroup's share and
around the chunks of rows dealt to the XCDs, and an X row of infinities and NaN, which may reach
only the rows that use it (lanes past a row's end read X row 0 and drop it)."""
import numpy as np
import pytest

from test_gpu_batch import TOL, run_spmm

import fastload_amd as fl

pytestmark = pytest.mark.gpu


def rows_matrix(m, n, seed):
    rng = np.random.default_rng(seed)
    lens = np.minimum(rng.choice([0, 1, 3, 4, 5, 15, 16, 17, 31, 32, 33, 40], m), n)
    rows = np.repeat(np.arange(m), lens)
    cols = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in lens] + [np.zeros(0, int)]).astype(np.int64)
    vals = rng.standard_normal(rows.size).astype(np.float32).astype(np.float64)
    o = np.lexsort((rows, cols))
    cp = np.concatenate([[0], np.cumsum(np.bincount(cols, minlength=n))]).astype(np.int32)
    return rows, cols, vals, (m, n, cp, rows[o].astype(np.int32), vals[o])


@pytest.mark.parametrize("kind", [fl.VAL_F64, fl.VAL_F32], ids=["f64", "f32"])
@pytest.mark.parametrize("k", [1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("m", [1, 15, 17, 64, 65, 1023, 1025, 9001])
def test_spmm_row_steps(gpu, m, k, kind):
    n = 53
    rows, cols, vals, csc = rows_matrix(m, n, 7 * m + k)
    M = fl.FastLoadMatrix(*csc, width=64)
    M.prepare_rows()
    X = np.random.default_rng(k).standard_normal((n, k)).astype(np.float32).astype(np.float64)
    want, scale = np.zeros((m, k)), np.zeros((m, k))
    np.add.at(want, rows, vals[:, None] * X[cols])
    np.add.at(scale, rows, np.abs(vals[:, None] * X[cols]))
    Y = run_spmm(M, X, kind, k)
    assert np.all(np.abs(Y - want) <= TOL[kind] * scale)  # empty rows: exactly 0
    X[0, ::2], X[0, 1::2] = np.inf, np.nan  # k = 1: inf
    uses = np.zeros(m, bool)
    uses[rows[cols == 0]] = True
    Z = run_spmm(M, X, kind, k)
    assert np.array_equal(Z[~uses], Y[~uses])
    assert not np.isfinite(Z[uses]).any()
