"""GPU test of the walks between columns and tiles (a wave takes 64 sorted columns and 32 depths, eight at a time
through LDS, in 16-byte pieces up to the arrays' end): column counts around groups of 64, column lengths
around the steps, the longest columns alone at the end. The layout must equal the oracle's bit for bit, and
the row order and the HYB split made from it must multiply right."""
import numpy as np
import pytest

from gpu_util import device_y, export_matches_oracle, rel_err
import oracle_bind as ob

import fastload_amd as fl
from fastload_amd import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 1000])
@pytest.mark.parametrize("lengths", ["steps", "one", "long_tail"])
@pytest.mark.parametrize("width", [32, 64])
def test_layout_edges(gpu, n, lengths, width):
    rng = np.random.default_rng(n + width)
    m = 700
    lens = {"steps": rng.choice([0, 1, 3, 4, 7, 8, 9, 31, 32, 33, 40, 64, 65, 100], n),
            "one": np.ones(n, int),
            "long_tail": np.where(np.arange(n) < max(1, n // 50), rng.integers(300, 700, n), rng.integers(0, 3, n))}[lengths]
    cp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ri = np.concatenate([np.sort(rng.choice(m, k, replace=False)) for k in lens]).astype(np.int32)
    v = rng.standard_normal(ri.size)
    x = rng.standard_normal(n)
    M = fl.FastLoadMatrix(m, n, cp, ri, v, width=width)
    bad, _ = export_matches_oracle(M, m, n, cp, ri, v, x, width)
    assert not bad
    want, scale = ob.spmv_oracle(m, n, cp, ri, v, x)
    M.prepare_rows()
    dy = DeviceArray(m, np.float64)
    M.spmm(DeviceArray.from_host(x), dy, 1, fl.VAL_F64)
    assert rel_err(dy.to_host(), want, scale) <= 1e-12
    for heavy in {0, min(n, 5), n}:
        M.prepare_hyb(heavy, 64, 1024)
        assert rel_err(device_y(M, x, fl.KERNEL_HYB, fl.VAL_F64), want, scale) <= 1e-12
