"""GPU test of FastLoad_spmv's repeated launches at row counts where all cleared copies of y fit at once,
where they are cleared in several groups, and where there is one: whole-number data, so y is exact."""
import numpy as np
import pytest

import fastload_amd as fl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 33, 41527, 41536, 60013, 2097153, 4194305])
def test_host_spmv(gpu, m):
    rng = np.random.default_rng(m)
    n = 300
    lengths = rng.integers(0, min(m, 40) + 1, n).astype(np.int32)
    colptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    row = np.concatenate([np.sort(rng.choice(m, k, replace=False)) for k in lengths]).astype(np.int32)
    val = rng.integers(-9, 10, len(row)).astype(np.float64)
    x = rng.integers(-9, 10, n).astype(np.float64)
    want = np.bincount(row, val * x[np.repeat(np.arange(n), lengths)], m)
    srow, sval, slen, sx, _ = fl.ColSort(m, n, lengths, colptr, row, val, x)
    tiles, _, _, _ = fl.formatTransform(srow, sval, slen, len(val), m, n)
    y, time_ms, _ = fl.FastLoad_spmv(tiles, len(val), n, m, sx)
    assert np.array_equal(y, want) and time_ms > 0
