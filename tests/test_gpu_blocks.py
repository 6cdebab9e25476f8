"""GPU test of the device memory that the library keeps from one matrix to the next: matrices of different
sizes made and dropped in turn by several threads, each on a stream of its own, with products still
running when their matrix is dropped; every product must be right."""
import threading

import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import DeviceArray, Stream

pytestmark = pytest.mark.gpu


def _work(seed, errors):
    try:
        s = Stream()
        for i in range(6):
            n = [3000, 20011, 3100, 60000, 2900, 59000][(i + seed) % 6]
            m, n, cp, ri, v = fl.gen_matrix(fl.GEN_ZIPF, 10 * seed + i, n, n, (1.9, 400))
            x = np.random.default_rng(i).standard_normal(n)
            cols = np.repeat(np.arange(n), np.diff(cp))
            want = np.bincount(ri, v * x[cols], m)
            scale = np.bincount(ri, np.abs(v * x[cols]), m)
            M = fl.FastLoadMatrix(m, n, cp, ri, v, width=64, stream=s)
            M.prepare_schedule(fl.KERNEL_PB, 128, 16384, stream=s)
            dx, dsx, dy = DeviceArray.from_host(x), DeviceArray(n, np.float64), DeviceArray(m, np.float64)
            M.permute_x(dx, dsx, stream=s)
            for _ in range(20):
                M.spmv(dsx, dy, fl.KERNEL_PB, fl.VAL_F64, stream=s, assign=True)
            M.close()  # the products may still be running
            assert np.all(np.abs(dy.to_host() - want) <= 1e-12 * scale)
    except Exception as e:  # noqa: BLE001
        errors.append(e)


@pytest.mark.parametrize("threads", [1, 4])
def test_blocks_threads_streams(gpu, threads):
    errors = []
    ts = [threading.Thread(target=_work, args=(k, errors)) for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors


def test_release_memory(gpu):
    """What a dropped matrix held is kept, serves the next of its size, and is given back on request; what is in use is not."""
    fl.release_memory()
    assert fl.release_memory() == 0
    m, n, cp, ri, v = fl.gen_matrix(fl.GEN_ZIPF, 5, 100_000, 100_000, (1.9, 400))

    def make():
        M = fl.FastLoadMatrix(m, n, cp, ri, v, width=64)
        M.prepare_schedule(fl.KERNEL_PB, 128, 16384)
        return M

    used = make()
    scratch = fl.release_memory()  # of the preparation
    assert scratch > 0
    other = make()
    fl.release_memory()
    other.close()
    kept = fl.release_memory()
    assert kept >= len(ri) * 12 + 8 * n  # values, rows and the column order at least
    x = np.random.default_rng(1).standard_normal(n)
    cols = np.repeat(np.arange(n), np.diff(cp))
    dx, dsx, dy = DeviceArray.from_host(x), DeviceArray(n, np.float64), DeviceArray(m, np.float64)
    used.permute_x(dx, dsx)
    used.spmv(dsx, dy, fl.KERNEL_PB, fl.VAL_F64, assign=True)
    scale = np.bincount(ri, np.abs(v * x[cols]), m)
    assert np.all(np.abs(dy.to_host() - np.bincount(ri, v * x[cols], m)) <= 1e-12 * scale)
    # a matrix that is dropped and made again takes the kept blocks: no more is kept than one matrix needs
    for _ in range(4):
        make().close()
    assert fl.release_memory() <= kept + 2 * scratch
