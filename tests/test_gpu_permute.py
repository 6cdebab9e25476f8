"""GPU test of fl_permute_x_*: sortx = x[perm] whatever the number of columns (the kernel moves
1,024 columns per workgroup, in groups of eight workgroups) and their lengths."""
import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 1023, 1024, 1025, 8191, 8192, 8193, 30011])
@pytest.mark.parametrize("loaded", [False, True])
def test_permute_x(gpu, n, loaded, tmp_path):
    rng = np.random.default_rng(n)
    lengths = np.minimum(rng.zipf(1.9, n), 60)
    cp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    ri = np.concatenate([np.sort(rng.choice(64, k, replace=False)) for k in lengths]).astype(np.int32)
    M = fl.FastLoadMatrix(64, n, cp, ri, rng.standard_normal(len(ri)), width=64)
    if loaded:
        M.save(str(tmp_path / "m"))
        M = fl.FastLoadMatrix.load(str(tmp_path / "m"))
    perm = M.perm()
    for dt in (np.float32, np.float64):
        x = rng.standard_normal(n).astype(dt)
        x[:: 7] = np.nan
        dsx = DeviceArray.zeros(n, dt)
        M.permute_x(DeviceArray.from_host(x), dsx)
        assert np.array_equal(dsx.to_host(), x[perm], equal_nan=True)
