"""GPU test: a solver whose matrix is prepared again between two solves into the same x (another batch size, band
height or heavy part; another schedule and back) uses the new arrays, as a solver made afterwards does."""
import numpy as np
import pytest
import scipy.sparse as sp

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu

AGAIN = {
    "win": (fl.KERNEL_WIN, [lambda M: M.prepare_schedule(fl.KERNEL_WIN, 256), lambda M: M.prepare_schedule(fl.KERNEL_WIN, 64),
                            lambda M: M.prepare_schedule(fl.KERNEL_WIN, 128)]),
    "win_and_back": (fl.KERNEL_WIN, [lambda M: M.prepare_schedule(fl.KERNEL_WIN, 256),
                                     lambda M: (M.prepare_schedule(fl.KERNEL_WINR, 64), M.prepare_schedule(fl.KERNEL_WIN, 256))]),
    "winr": (fl.KERNEL_WINR, [lambda M: M.prepare_schedule(fl.KERNEL_WINR, 64), lambda M: M.prepare_schedule(fl.KERNEL_WINR, 256)]),
    "pb": (fl.KERNEL_PB, [lambda M: M.prepare_schedule(fl.KERNEL_PB, 64, 1024), lambda M: M.prepare_schedule(fl.KERNEL_PB, 256, 16384),
                          lambda M: M.prepare_schedule(fl.KERNEL_PB, 256, 1024)]),
    "hyb": (fl.KERNEL_HYB, [lambda M: M.prepare_hyb(500, 128, 16384), lambda M: M.prepare_hyb(5000, 64, 1024),
                            lambda M: M.prepare_hyb(0, 128, 4096)]),
}


@pytest.mark.parametrize("name", list(AGAIN))
@pytest.mark.parametrize("kind", [fl.VAL_F64, fl.VAL_F32], ids=["f64", "f32"])
def test_cg_after_preparing_again(gpu, name, kind):
    rng = np.random.default_rng(3)
    n = 20_011
    i, j = rng.integers(0, n, 6 * n), rng.integers(0, n, 6 * n)
    B = sp.coo_matrix((rng.uniform(-1, 1, len(i)), (i, j)), shape=(n, n))
    B = sp.csc_matrix(B + B.T)
    B *= 2.0 / abs(B).sum(axis=1).max()
    A = sp.csc_matrix(B + 4.0 * sp.identity(n))  # the eigenvalues lie in [2, 6]
    A.sort_indices()
    dt, rtol = (np.float64, 1e-12) if kind == fl.VAL_F64 else (np.float32, 1e-5)
    kernel, ways = AGAIN[name]
    M = fl.FastLoadMatrix(n, n, A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data, width=64)
    M.prepare(kind)
    cg, dx = None, DeviceArray.zeros(n, dt)
    for way in ways:
        way(M)
        cg = cg or fl.CG(M, kernel, kind)
        for solver in (cg, fl.CG(M, kernel, kind)):
            b = (A @ rng.standard_normal(n)).astype(dt)
            dx.zero()
            it, res = solver.solve(DeviceArray.from_host(b), dx, max_iter=100, rtol=rtol, check_every=4)
            # kappa <= 3: the error falls by 0.27 or more per iteration, 2 * 0.27^k <= 1e-12 at k = 22
            assert it <= (24 if kind == fl.VAL_F64 else 16) and res <= rtol
            true = np.linalg.norm(b - A @ dx.to_host().astype(np.float64))
            assert true <= (rtol + 100 * np.finfo(dt).eps) * np.linalg.norm(b)
