"""The band heights that PB runs with: fl_band_rows against the rule (at most what is asked for, every compute unit a band,
32 products of a batch to each), and the selector's classes that are the same schedule on a matrix."""
import numpy as np
import pytest

import fastload_amd as fl
from fastload_amd import selector as sel


@pytest.mark.parametrize("bt", [64, 128, 256])
@pytest.mark.parametrize("most", [1024, 4096, 16384])
def test_band_rows(bt, most):
    for m in (0, 1, 1024, 131_072, 131_073, 262_144, 262_145, 1_048_576, 1_048_577, 4_194_304, 4_194_305, 2**31 - 1):
        bands = min(256, 2 * bt)
        low = max(1024, -(-(-(-m // bands)) // 1024) * 1024)
        assert fl.band_rows(m, bt, most) == min(most, low)


def test_band_rows_refuses():
    for m, bt, most in ((-1, 128, 4096), (5, 100, 4096), (5, 128, 1023), (5, 128, 16385)):
        with pytest.raises(fl.FastLoadError):
            fl.band_rows(m, bt, most)


def test_same_schedules():
    name = {s.name: c for c, s in enumerate(sel.SCHEDULES)}
    low = {c: sel.effective(c, 1_048_576) for c in range(sel.N_CLASSES)}
    assert len(set(low.values())) == sel.N_CLASSES - 3
    assert low[name["pb128_r4k"]] == low[name["pb128_r16k"]] != low[name["pb256_r16k"]]
    assert low[name["pb256_r4k"]] == low[name["pb256_r8k"]] == low[name["pb256_r16k"]]
    assert len({sel.effective(c, 8_000_000) for c in range(sel.N_CLASSES)}) == sel.N_CLASSES


@pytest.mark.gpu
def test_choose_refined_times_a_schedule_once(gpu, monkeypatch):
    m, n, cp, ri, v = fl.gen_matrix(fl.GEN_ZIPF, 5, 20_000, 20_000, (1.9, 400))
    d = [fl.DeviceArray.from_host(a) for a in (cp, ri, v)]
    calls = []

    def timer(step, dy, **kw):
        calls.append(step)
        return float(len(calls))

    monkeypatch.setattr(sel, "time_schedule", timer)
    s = sel.Selector()
    c, times, f = s.choose_refined(m, n, *d, top=sel.N_CLASSES)
    assert set(times) == set(range(sel.N_CLASSES)) and len(calls) == sel.N_CLASSES - 3
    for a in times:
        for b in times:
            assert (times[a] == times[b]) == (sel.effective(a, m) == sel.effective(b, m))
    assert c == s.rank_features(f)[0] and np.isfinite(f).all()
