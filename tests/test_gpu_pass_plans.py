"""Which lattices run in passes of several calls (lbmc_pass_info), and the
smallest margin, one node, in every kernel: bit for bit as one call per launch."""
import numpy as np
import pytest

import cases
from test_gpu_passes import D2_CASES, D3_CASES

pytestmark = pytest.mark.gpu
lbmc = pytest.importorskip("lbmc")


def _built(monkeypatch, case, storage, shape):
    if shape is None:
        monkeypatch.delenv("LBMC_PASS", raising=False)
    else:
        monkeypatch.setenv("LBMC_PASS", shape)
    return cases.build(lbmc.Lattice, case, storage=storage)


def _calls(lat):
    return lat.pass_info()["calls"]


def _ran(lat, store_every):
    lat.run(3, 23, store_every)
    lat.run(26, 13, 4)
    rho, u = lat.get_macros()
    out = lat.get_f(), rho, u
    lat.close()
    return out


@pytest.mark.parametrize("storage", [0, 1, 2, 3], ids=["f64", "f32", "f16s", "bf16s"])
@pytest.mark.parametrize("case", D2_CASES, ids=lambda c: c["name"])
def test_smallest_margin(monkeypatch, case, storage):
    for store_every in (0, 5):
        lat = _built(monkeypatch, case, storage, "0")
        assert _calls(lat) == 1
        want = _ran(lat, store_every)
        for shape in ("0,16,16,1", "0,3,3,1", "1,64,8,1", "2,64,16,1", "2,17,57,1"):
            lat = _built(monkeypatch, case, storage, shape)
            assert _calls(lat) == 2, shape
            for a, b in zip(_ran(lat, store_every), want):
                assert np.array_equal(a, b), (shape, store_every)


@pytest.mark.parametrize("storage", [0, 1, 2, 3], ids=["f64", "f32", "f16s", "bf16s"])
def test_plans_of_d2q9(monkeypatch, storage):
    for case in D2_CASES:
        lat = _built(monkeypatch, case, storage, None)
        info = lat.pass_info()
        assert info["calls"] > 1 and min(info["width"], info["height"]) > 2 * (info["calls"] - 1), case["name"]
        lat.close()
        # a margin of none is no pass
        lat = _built(monkeypatch, case, storage, "0,16,16,0")
        assert _calls(lat) == 1
        lat.close()
    # 16-bit lattices above 2^20 nodes, and sf faces, go one call per launch
    lat = _built(monkeypatch, cases.channel_d2q9(1031, 1021), storage, None)
    assert (_calls(lat) == 1) == (storage >= 2)
    lat.close()
    lat = _built(monkeypatch, cases.sf_d2q9(), storage, None)
    assert _calls(lat) == 1
    lat.close()


@pytest.mark.parametrize("storage", [0, 1, 2], ids=["f64", "f32", "f16s"])
def test_plans_of_d3q15(monkeypatch, storage):
    for case in D3_CASES:
        for shape in ("37,13,3", "9,7,2", "3,3,64", "64,8,1"):
            lat = _built(monkeypatch, case, storage, shape)
            passes = storage < 2 and not case["name"].startswith("faces")
            assert _calls(lat) == (2 if passes else 1), (case["name"], shape)
            lat.close()
    n = 131 * 96 * 75
    lat = lbmc.Lattice(lbmc.D3Q15, (131, 96, 75), tau=0.6, storage=storage)
    monkeypatch.delenv("LBMC_PASS", raising=False)
    lat.set_fields(geometry=np.zeros(n))
    assert _calls(lat) == (2 if storage < 2 else 1)
    lat.close()


def test_members_of_a_batch_hold_their_buffers(monkeypatch):
    # what the comparisons of batches in passes rest on
    for case in D2_CASES:
        for storage in (0, 1):
            lat = _built(monkeypatch, case, storage, None)
            batch = lbmc.Batch([lat])
            batch.run(0, 9, 0)
            assert _calls(lat) > 1
            batch.close()
            lat.close()


@pytest.mark.parametrize("storage", [0, 1, 2, 3], ids=["f64", "f32", "f16s", "bf16s"])
@pytest.mark.parametrize("case", [cases.channel_d2q9(300, 200), cases.pressure_d2q9(Lx=300, Ly=200),
                                  cases.channel_d2q9(1148, 450), cases.pressure_d2q9(Lx=61, Ly=47)],
                         ids=lambda c: c["name"])
def test_runs_of_every_length(monkeypatch, case, storage):
    """Every number of calls around the lengths of a pass, with the tiles of
    each, and stretches of every length between stored prescribed values."""
    out = []
    for shape in ("0", None):
        lat = _built(monkeypatch, case, storage, shape)
        assert (_calls(lat) == 1) == (shape == "0")
        t = 0
        for n in range(1, 19):
            lat.run(t, n, 0)
            t += n
        for store_every in range(1, 11):
            lat.run(t, 23, store_every)
            t += 23
        rho, u = lat.get_macros()
        out.append((lat.get_f(), rho, u))
        lat.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
