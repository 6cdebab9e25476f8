"""GPU test of Selector.choose against fl_select_schedule: with and without a network, for an empty
matrix, below the probability limit, and with a network of other dimensions."""
import ctypes as C

import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray
from fastload_amd import selector as sel

pytestmark = pytest.mark.gpu


def _matrix(m, n, per, rng):
    lengths = rng.integers(0, per + 1, n)
    cp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    ri = np.concatenate([np.sort(rng.choice(m, k, replace=False)) for k in lengths]).astype(np.int32)
    return DeviceArray.from_host(cp), DeviceArray.from_host(ri) if len(ri) else None


@pytest.mark.parametrize("m,n,per", [(5, 3, 2), (1000, 700, 12), (400, 9000, 3), (10, 10, 0)])
@pytest.mark.parametrize("weights", [sel.WEIGHTS_PATH, None])
def test_choose_is_select_schedule(gpu, m, n, per, weights):
    dcp, dri = _matrix(m, n, per, np.random.default_rng(m + n))
    s = sel.Selector(weights)
    c, p, f = s.choose(m, n, dcp, dri)
    out, pr = C.c_int(7), C.c_float(1.0)
    rc = fl.lib.fl_select_schedule(s.mlp.handle if s.mlp else None, m, n, dri.count if dri else 0, dcp.ptr,
                                   dri.ptr if dri else None, C.byref(out), C.byref(pr), None)
    assert rc == 0 and out.value == c
    # the features are sums in an order that changes: a rounding of FP32 each, amplified by the network
    assert abs(pr.value - p) <= 1e-5
    assert np.allclose(f, sel.features(m, n, dcp, dri), rtol=1e-6, atol=0)
    if s.mlp is None or not dri:
        assert (c, p) == (sel.DEFAULT_CLASS, 0.0)
    strict = sel.Selector(weights, min_prob=1.1)
    assert strict.choose(m, n, dcp, dri)[0] == sel.DEFAULT_CLASS


def test_choose_refuses_other_networks(gpu):
    dcp, dri = _matrix(100, 100, 4, np.random.default_rng(1))
    s = sel.Selector(None)
    s.mlp = sel.MLP((sel.N_FEATURES, 8, 8, 3))
    with pytest.raises(fl.FastLoadError) as e:
        s.choose(100, 100, dcp, dri)
    assert e.value.rc == -8
