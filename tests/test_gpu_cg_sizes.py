"""GPU test of the solver's vector kernels at row counts around their blocks (256 blocks of 512 threads, a
contiguous range each): tridiagonal systems, with schedules that add to a cleared q, that write it, and
that read p in the original order; and a second solve with a longer replay group."""
import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 255, 257, 511, 131071, 131073, 300007])
@pytest.mark.parametrize("kernel", [fl.KERNEL_WINR, fl.KERNEL_PB, fl.KERNEL_ROW, fl.KERNEL_DROPIN],
                         ids=["winr", "pb", "row", "dropin"])
def test_cg_sizes(gpu, n, kernel):
    i = np.arange(n)
    rows = np.stack([i - 1, i, i + 1], 1)
    vals = np.tile([-1.0, 4.0, -1.0], (n, 1))
    keep = (rows >= 0) & (rows < n)
    cp = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    M = fl.FastLoadMatrix(n, n, cp, rows[keep].astype(np.int32), vals[keep], width=64)
    if kernel == fl.KERNEL_ROW:
        M.prepare_rows()
    elif kernel != fl.KERNEL_DROPIN:
        M.prepare_schedule(kernel, 64, 16384)
    rng = np.random.default_rng(n)
    cg = fl.CG(M, kernel, fl.VAL_F64)
    for every in (10, 24):
        want = rng.standard_normal(n)
        b = 4.0 * want
        b[1:] -= want[:-1]
        b[:-1] -= want[1:]
        dx = DeviceArray.zeros(n, np.float64)
        it, res = cg.solve(DeviceArray.from_host(b), dx, max_iter=200, rtol=1e-12, check_every=every)
        assert it % every == 0 and it <= 72 and res <= 1e-12
        # A has its eigenvalues in [2, 6]: |x - want| <= |b - A x| / 2
        assert np.linalg.norm(dx.to_host() - want) <= 1e-12 * np.linalg.norm(b)
