"""GPU test of fl_features from 2^20 entries on, where the row counts come from grouped indices: row
counts around the 256 groups and their widths, groups cut by the counting chunks of 65,536 entries, all
entries in one row, empty rows, and more rows than the grouped path takes."""
import numpy as np
import pytest

from oracle import selector_oracle as so

from fastload_amd import DeviceArray
from fastload_amd import selector as sel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,rows", [(1, "all"), (200, "all"), (257, "all"), (70000, "all"), (70000, "one"),
                                    (1 << 20, "half"), (8388608, "all"), (8388609, "all")])
def test_features_large(gpu, m, rows):
    rng = np.random.default_rng(m)
    n = (1 << 20) + 77
    ri = {"all": lambda: rng.integers(0, m, n), "one": lambda: np.full(n, m - 3),
          "half": lambda: rng.integers(m // 4, m // 2, n)}[rows]().astype(np.int32)
    lens = np.ones(n, np.int64)
    lens[1000:1400] = 0  # some empty columns, their entries in a longer one
    lens[1400] = 401
    ri[1000:1401] = np.sort(ri[1000:1401])
    cp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    f = sel.features(m, n, DeviceArray.from_host(cp), DeviceArray.from_host(ri))
    want = so.features(m, n, cp, ri)
    assert np.allclose(f, want, rtol=2e-6, atol=1e-7)  # FP64 sums rounded to FP32
