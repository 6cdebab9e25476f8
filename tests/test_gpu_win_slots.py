"""GPU test of the WIN and WINR schedules' slots, row lists and marks of shared rows against their definition
in numpy, at the edges of the bitmap that counts a batch's rows (262,144 rows, of which up to 16 for rows
anywhere in the matrix) and above them, where the entries are sorted. Exact."""
import numpy as np
import pytest

import fastload_amd as fl
from flmx_util import sections

pytestmark = pytest.mark.gpu

SEG = 1 << 18


@pytest.mark.parametrize("m", [1, 3001, SEG, SEG + 1, 5 * SEG + 3, 16 * SEG, 16 * SEG + 1])
@pytest.mark.parametrize("n,exponent", [(70, 2.5), (5001, 1.7)])
@pytest.mark.parametrize("bt", [64, 128, 256])
@pytest.mark.parametrize("kernel", [fl.KERNEL_WIN, fl.KERNEL_WINR], ids=["win", "winr"])
def test_slots(gpu, tmp_path, m, n, exponent, bt, kernel):
    rng = np.random.default_rng(m + n)
    lens = np.minimum(np.minimum(rng.zipf(exponent, n), 900), m)
    rows = np.concatenate([np.sort(rng.choice(m, k, replace=False) if m <= SEG else  # distinct: one per part
                                   np.arange(k) * (m // k) + rng.integers(0, m // k, k)) for k in lens])
    rows[np.cumsum(lens) - 1] = m - 1  # the last row gets an entry of every column
    cp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    M = fl.FastLoadMatrix(m, n, cp, rows.astype(np.int32), np.ones(rows.size), width=64)
    M.prepare_schedule(kernel, bt, 16384)
    M.save(str(tmp_path / "m.flmx"))
    raw = (tmp_path / "m.flmx").read_bytes()
    sec = sections(raw)
    slot, lists, off = (np.frombuffer(raw, dt, sec[t][2], sec[t][3]) for t, dt in
                        ((20, np.uint16), (21, np.int32), (22, np.int32)))
    e = M.export()
    ptr, row, col = e["tile_ptr"][:-1], e["sortrowidx"].astype(np.int64), e["tile_colidx"]
    batch = np.empty(row.size, np.int64)
    key = row[ptr] >> 6 if kernel == fl.KERNEL_WINR else col >> 8
    for i, t in enumerate(np.argsort(key, kind="stable")):
        batch[ptr[t]:ptr[t] + min(64, n - col[t])] = i // bt
    nb = -(-ptr.size // bt)
    pairs, place = np.unique(batch * m + row, return_inverse=True)
    want_off = np.searchsorted(pairs // m, np.arange(nb + 1))
    want_rows, times = pairs % m, np.bincount(np.searchsorted(np.unique(pairs % m), pairs % m))
    shared = times[np.searchsorted(np.unique(pairs % m), pairs % m)] > 1
    assert np.array_equal(off, want_off)
    assert np.array_equal(slot, place - want_off[batch])
    assert np.array_equal(lists & 0x7fffffff, want_rows)
    assert np.array_equal(lists < 0, shared)
