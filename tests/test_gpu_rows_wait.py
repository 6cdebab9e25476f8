"""GPU test: fl_matrix_prepare_rows returns with the row order written, also for a matrix without entries (its row
pointers are only cleared), so a product on another stream may follow at once."""
import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray, Event, Stream
from fastload_amd._lib import check, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nnz", [0, 3])
def test_rows_are_ready_on_return(gpu, nnz):
    m, n = 70_001, 64
    cp = np.zeros(n + 1, np.int32)
    cp[1:] = nnz
    M = fl.FastLoadMatrix(m, n, cp, np.arange(nnz, dtype=np.int32), np.ones(nnz), width=64)
    busy, other = Stream(), Stream()
    ahead = DeviceArray(1 << 32, np.uint8)  # fills of 4 GiB: about a millisecond each of work queued before the preparation
    x, y = DeviceArray.from_host(np.ones(n, np.float32)), DeviceArray.from_host(np.full(m, 7, np.float32))
    before, after = Event(), Event()
    for _ in range(8):
        check(lib.fl_zero_device(ahead.ptr, ahead.nbytes, busy.ptr), "fl_zero_device")
    before.record(busy)
    M.prepare_rows(stream=busy)
    M.spmm(x, y, 1, fl.VAL_F32, stream=other)
    after.record(other)
    assert before.elapsed_ms(after) >= 0.0  # the product began when the queued fills had ended
    want = np.zeros(m, np.float32)
    want[:nnz] = 1
    assert np.array_equal(y.to_host(), want)
