"""GPU test of the row kernels on matrices with a row much longer than the others: every k, both value kinds, X and Y at
addresses for 16-byte lanes and narrower ones, rows that end at the edges of steps and groups next to one of 1,000 entries. The kernel is chosen by the whole matrix, so the same
rows above rows of 600 entries, where the long one is none, have to give the same bits."""
import time

import numpy as np
import pytest

from test_gpu_batch import TOL

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu

N = 1100
LENS = [0, 1, 2, 3, 4, 5, 11, 12, 13, 15, 16, 17, 31, 32, 33, 47, 48, 49, 51, 52, 53, 63, 64, 65, 67, 68, 69, 113, 127, 128, 129]


def _matrix(m, n, rows, cols, vals):
    o = np.lexsort((rows, cols))
    cp = np.concatenate([[0], np.cumsum(np.bincount(cols, minlength=n))]).astype(np.int32)
    M = fl.FastLoadMatrix(m, n, cp, rows[o].astype(np.int32), vals[o], width=64)
    M.prepare_rows()
    return M


def _product(M, X, Y, k, kind, accumulate, shift):
    dt = np.float64 if kind == fl.VAL_F64 else np.float32

    def put(a):  # `shift` elements from the start of an allocation
        return DeviceArray.from_host(np.r_[np.zeros(shift, dt), a.astype(dt).ravel()]).view(shift, a.size)

    dx, dy = put(X), put(Y)
    M.spmm(dx, dy, k, kind, accumulate=accumulate)
    return dy.to_host().reshape(-1, k)


@pytest.fixture(scope="module")
def pair(gpu):
    """(rows, cols, vals) of 3,000 short rows and a long one, and the matrices alone and above long rows."""
    rng = np.random.default_rng(1)
    m = 3001
    lens = rng.integers(0, 4, m)
    lens[:: m // len(LENS)][: len(LENS)] = LENS
    lens[1733] = 1000
    rows = np.repeat(np.arange(m), lens)
    cols = np.concatenate([np.sort(rng.choice(N, c, replace=False)) for c in lens])
    vals = rng.standard_normal(rows.size).astype(np.float32).astype(np.float64)
    rows2 = np.repeat(np.arange(m, 2 * m), 600)
    cols2 = np.tile(np.arange(N, N + 600), m)
    both = _matrix(2 * m, 2 * N, np.r_[rows, rows2], np.r_[cols, cols2], np.r_[vals, np.ones(rows2.size)])
    return m, rows, cols, vals, _matrix(m, N, rows, cols, vals), both


@pytest.mark.parametrize("kind", [fl.VAL_F64, fl.VAL_F32], ids=["f64", "f32"])
@pytest.mark.parametrize("k", [1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("shift", [0, 1, 2])
def test_long_row_among_short_ones(pair, k, kind, shift):
    m, rows, cols, vals, alone, both = pair
    rng = np.random.default_rng(k)
    X = rng.standard_normal((2 * N, k)).astype(np.float32).astype(np.float64)
    Y = rng.standard_normal((2 * m, k)).astype(np.float32).astype(np.float64)
    want, scale = np.zeros((m, k)), np.zeros((m, k))
    np.add.at(want, rows, vals[:, None] * X[cols])
    np.add.at(scale, rows, np.abs(vals[:, None] * X[cols]))
    for accumulate in (False, True):
        a = _product(alone, X[:N], Y[:m], k, kind, accumulate, shift)
        more = Y[:m] if accumulate else 0.0
        assert np.all(np.abs(a - (want + more)) <= TOL[kind] * (scale + np.abs(more)))
        assert np.array_equal(a, _product(both, X, Y, k, kind, accumulate, shift)[:m])
    # an X row of infinities reaches only the rows that use it
    Z = X.copy()
    Z[0] = np.inf
    uses = np.zeros(m, bool)
    uses[rows[cols == 0]] = True
    b = _product(alone, Z[:N], Y[:m], k, kind, False, shift)
    assert np.array_equal(b[~uses], _product(alone, X[:N], Y[:m], k, kind, False, shift)[~uses]) and not np.isfinite(b[uses]).any()


@pytest.mark.parametrize("k,most", [(1, 0.4), (2, 1.4), (8, 2.0), (32, 2.6)])
def test_time_of_one_long_row(gpu, k, most):
    """50,000 entries in one row, FP32, ms: 0.2, 0.7, 0.8, 1.2 for k = 1, 2, 8, 32; with two lanes for k = 1 and four X rows
    in flight 0.63, 1.6, 3.4, 4.1."""
    m, n = 20_000, 100_000
    rng = np.random.default_rng(2)
    rows = np.r_[np.repeat(np.arange(m), 3), np.full(50_000, 777)]
    M = _matrix(m, n, rows, rng.integers(0, n, rows.size), np.ones(rows.size))
    X, Y = DeviceArray.zeros(n * k, np.float32), DeviceArray.zeros(m * k, np.float32)
    best = np.inf
    for _ in range(5):
        fl.synchronize()
        t = time.perf_counter()
        for _ in range(10):
            M.spmm(X, Y, k, fl.VAL_F32)
        fl.synchronize()
        best = min(best, (time.perf_counter() - t) / 10)
    assert best * 1e3 < most


def test_long_row_from_a_file(pair, tmp_path):
    """The row order read back: the same kernel, the same bits."""
    m, rows, cols, vals, alone, _ = pair
    alone.save(tmp_path / "hub.flmx")
    loaded = fl.FastLoadMatrix.load(tmp_path / "hub.flmx")
    for k in (1, 2, 8):
        X, Y = np.random.default_rng(k).standard_normal((N, k)), np.zeros((m, k))
        args = X, Y, k, fl.VAL_F64, False, 0
        assert np.array_equal(_product(alone, *args), _product(loaded, *args))
