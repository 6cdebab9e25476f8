"""GPU test of the PB schedule's places, staging slots and runs against their definition in numpy: one band,
the edges of the bands that a workgroup counts in LDS (4,096, and one more, where the entries are
sorted), a few entries for many bands, and batches that end inside a group of eight. Exact."""
import numpy as np
import pytest

import fastload_amd as fl
from flmx_util import sections

pytestmark = pytest.mark.gpu

TAGS = {30: np.uint16, 31: np.uint16, 32: np.int32, 33: np.int32, 34: np.int32, 35: np.int32, 36: np.int32}


def places(m, n, e, bt, asked):
    """The sections 30 to 36 of a matrix with one chunk, from its tile layout."""
    ptr, rows, col = e["tile_ptr"][:-1], e["sortrowidx"], e["tile_colidx"]
    R = min(asked, max(1024, -(-(-(-m // min(256, 2 * bt))) // 1024) * 1024))
    nbands = max(-(-m // R), 1)
    batch = np.empty(rows.size, np.int64)
    for i, t in enumerate(np.argsort(col >> 8, kind="stable")):
        batch[ptr[t]:ptr[t] + min(64, n - col[t])] = i // bt
    nb = -(-ptr.size // bt)
    band = rows // R
    order = np.lexsort((np.arange(rows.size), batch >> 3, batch & 7, band))  # band, batch in XCD order, entry
    place = np.empty(rows.size, np.int64)
    place[order] = np.arange(rows.size)
    by = np.lexsort((np.arange(rows.size), band, batch))
    start = np.searchsorted(batch[by], np.arange(nb + 1))
    slot = np.empty(rows.size, np.int64)
    slot[by] = np.arange(rows.size) - start[batch[by]]
    key = (batch * nbands + band)[by]
    head = np.flatnonzero(np.r_[True, key[1:] != key[:-1]])
    return {30: slot, 31: (rows % R)[order], 32: np.searchsorted(band[order], np.arange(nbands + 1)),
            33: np.searchsorted(batch[by][head], np.arange(nb + 1)), 34: slot[by[head]], 35: place[by[head]],
            36: np.diff(np.r_[head, rows.size])}


@pytest.mark.parametrize("m,asked", [(1, 16384), (1024, 16384), (1025, 16384), (66001, 16384), (300007, 1500),
                                     (4096 * 1024, 1024), (4096 * 1024 + 1, 1024)])
@pytest.mark.parametrize("n,exponent", [(70, 2.5), (5001, 1.7)])
@pytest.mark.parametrize("bt", [64, 256])
def test_places(gpu, tmp_path, m, asked, n, exponent, bt):
    rng = np.random.default_rng(m + n)
    lens = np.minimum(np.minimum(rng.zipf(exponent, n), 900), m)
    rows = np.concatenate([np.sort(rng.choice(m, k, replace=False)) for k in lens]).astype(np.int32)
    cp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    M = fl.FastLoadMatrix(m, n, cp, rows, np.ones(rows.size), width=64)
    M.prepare_schedule(fl.KERNEL_PB, bt, asked)
    M.save(str(tmp_path / "m.flmx"))
    raw = (tmp_path / "m.flmx").read_bytes()
    sec = sections(raw)
    for tag, want in places(m, n, M.export(), bt, asked).items():
        _, elem, count, off, _ = sec[tag]
        got = np.frombuffer(raw, TAGS[tag], count, off)
        assert elem == got.itemsize and np.array_equal(got, want), tag
