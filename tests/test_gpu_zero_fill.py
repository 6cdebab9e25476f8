"""GPU test of the zero fill: sizes around 4 and 16 bytes and a workgroup, from 16-byte and 4-byte aligned
addresses; nothing outside the range is written."""
import numpy as np
import pytest

from fastload_amd import DeviceArray
from fastload_amd._lib import check, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bytes_", [0, 1, 3, 4, 5, 15, 16, 17, 20, 31, 4095, 4096, 4099, 364500, 1048580])
@pytest.mark.parametrize("offset", [0, 4, 16, 20])
def test_zero_fill(gpu, bytes_, offset):
    host = np.full(offset + bytes_ + 64, 7, np.uint8)
    d = DeviceArray.from_host(host)
    check(lib.fl_zero_device(d.ptr.value + offset if hasattr(d.ptr, "value") else d.ptr + offset, bytes_, None), "fl_zero_device")
    host[offset:offset + bytes_] = 0
    assert np.array_equal(d.to_host(), host)
