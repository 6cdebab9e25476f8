"""GPU test of the solver where the WIN and WINR products also sum p . q: every batch size (and with it
both block sizes), both value kinds, rows owned by one batch and shared by several, more slots than
threads, and a matrix with an empty row and column. A = 4 I + B with |eigenvalues of B| <= 2, so that
|x - want| <= |b - A x| / 2."""
import numpy as np
import pytest
import scipy.sparse as sp

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu


def _system(pattern, n, rng):
    if pattern == "band":  # neighbours within 64 rows: mostly owned rows
        i = np.repeat(np.arange(n), 4)
        j = np.clip(i + rng.integers(-64, 65, len(i)), 0, n - 1)
    else:  # anywhere: shared rows, a slot for almost every entry
        i, j = rng.integers(0, n, 5 * n), rng.integers(0, n, 5 * n)
    B = sp.coo_matrix((rng.uniform(-1, 1, len(i)), (i, j)), shape=(n, n))
    B = sp.csc_matrix(B + B.T)
    B *= 2.0 / max(abs(B).sum(axis=1).max(), 1e-30)
    A = sp.csc_matrix(B + 4.0 * sp.identity(n))
    A.sort_indices()
    return A


@pytest.mark.parametrize("kernel", [fl.KERNEL_WIN, fl.KERNEL_WINR], ids=["win", "winr"])
@pytest.mark.parametrize("bt", [64, 128, 256])
@pytest.mark.parametrize("kind", [fl.VAL_F64, fl.VAL_F32], ids=["f64", "f32"])
@pytest.mark.parametrize("pattern,n", [("band", 70), ("band", 30011), ("anywhere", 1000), ("anywhere", 40009)])
def test_cg_with_dot(gpu, kernel, bt, kind, pattern, n):
    rng = np.random.default_rng(n + bt)
    A = _system(pattern, n, rng)
    M = fl.FastLoadMatrix(n, n, A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data, width=64)
    dt, rtol = (np.float64, 1e-12) if kind == fl.VAL_F64 else (np.float32, 1e-5)
    M.prepare(kind)
    M.prepare_schedule(kernel, bt)
    cg = fl.CG(M, kernel, kind)
    for _ in range(2):
        want = rng.standard_normal(n)
        b = (A @ want).astype(dt)
        dx = DeviceArray.zeros(n, dt)
        it, res = cg.solve(DeviceArray.from_host(b), dx, max_iter=100, rtol=rtol, check_every=4)
        # kappa <= 3: the error falls by 0.27 or more per iteration, 2 * 0.27^k <= 1e-12 at k = 22
        assert it <= (24 if kind == fl.VAL_F64 else 16) and res <= rtol
        # the recursive residual and b - A x part by a few roundings per iteration
        true = np.linalg.norm(b - A @ dx.to_host().astype(np.float64))
        assert true <= (rtol + 100 * np.finfo(dt).eps) * np.linalg.norm(b)


def test_cg_with_dot_empty_row(gpu):
    """p . q = 0 parts and rows no batch owns: the empty row's residual stays, the others are solved."""
    n = 200
    A = sp.lil_matrix(4.0 * sp.identity(n))
    A[7, 7] = 0.0
    A = sp.csc_matrix(A)
    A.eliminate_zeros()
    M = fl.FastLoadMatrix(n, n, A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data, width=64)
    M.prepare_schedule(fl.KERNEL_WINR, 64)
    b = np.arange(1.0, n + 1)
    b[7] = 0.0
    dx = DeviceArray.zeros(n, np.float64)
    it, res = fl.CG(M, fl.KERNEL_WINR, fl.VAL_F64).solve(DeviceArray.from_host(b), dx, max_iter=10, rtol=1e-12,
                                                         check_every=2)
    assert it == 2 and res <= 1e-12 and np.abs(dx.to_host() - b / 4).max() <= 1e-12
