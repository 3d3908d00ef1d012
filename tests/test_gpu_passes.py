"""Passes of several calls (lbmc_run on D2Q9 lattices) against one call per
launch, bit for bit: the same node updates in another order of memory traffic.
LBMC_PASS=0 keeps one call per launch, "size,W,H,M" forces a tile shape."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu
lbmc = pytest.importorskip("lbmc")

D2_CASES = [
    cases.channel_d2q9(32, 16),
    cases.channel_d2q9(131, 65, collision=cases.MRT, rates=cases.d2q9_rates(0.8)),
    cases.channel_d2q9(3, 5),                       # smaller than the tile and its margin
    cases.pressure_d2q9(porous=True, collision=cases.MRTPOR),  # prescribed values, Zou-He, porous
    cases.pressure_d2q9(collision=cases.BGK),
    cases.porous_d2q9(L=70, collision=cases.NTPOR),
]


def _run(monkeypatch, case, storage, shape, store_every, t0=3):
    if shape is None:
        monkeypatch.delenv("LBMC_PASS", raising=False)
    else:
        monkeypatch.setenv("LBMC_PASS", shape)
    lat = cases.build(lbmc.Lattice, case, storage=storage)
    # whole passes, a remainder, a lone call, then a run that starts from the
    # stored layout of another call
    lat.run(t0, 23, store_every)
    lat.run(t0 + 23, 2, 7)
    lat.step(t0 + 25, False)
    lat.run(t0 + 26, 12, 4)
    rho, u = lat.get_macros()
    out = lat.get_f(), rho, u
    lat.close()
    return out


@pytest.mark.parametrize("storage", [0, 1, 2, 3], ids=["f64", "f32", "f16s", "bf16s"])
@pytest.mark.parametrize("case", D2_CASES, ids=lambda c: c["name"])
def test_passes_match_one_call_per_launch(monkeypatch, case, storage):
    for store_every in (0, 1, 5):
        want = _run(monkeypatch, case, storage, "0", store_every)
        # the planned shape; every kernel size with its smallest, an uneven and
        # its deepest margin
        for shape in (None, "0,16,16,0", "0,16,16,7", "1,32,16,5", "2,64,16,2", "2,17,57,6", "2,1,1,0"):
            got = _run(monkeypatch, case, storage, shape, store_every)
            for a, b in zip(got, want):
                assert np.array_equal(a, b), (shape, store_every)


def test_long_time_index_and_late_start(monkeypatch):
    case = cases.channel_d2q9(37, 21)
    want = _run(monkeypatch, case, 0, "0", 3, t0=2 ** 31 + 5)
    got = _run(monkeypatch, case, 0, None, 3, t0=2 ** 31 + 5)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
