"""Batches beyond the sizes below which runs go one call per launch
(batch_passes): members of every kind in passes against one call per launch,
bit for bit."""
import numpy as np
import pytest

import cases
import pymlp

pytestmark = pytest.mark.gpu
lbmc = pytest.importorskip("lbmc")


def _group(prescribed):
    g = [cases.channel_d2q9(701, 397, collision=cases.MRT, rates=cases.d2q9_rates(0.8)), cases.channel_d2q9(1031, 613),
         cases.porous_d2q9(L=401, collision=cases.NTPOR), cases.channel_d2q9(512, 256), cases.channel_d2q9(90, 31)]
    return g + [cases.pressure_d2q9(Lx=301, Ly=199)] * prescribed


def _stepped(monkeypatch, path, group, storage, every, store_every, runs):
    if path:
        monkeypatch.setenv("LBMC_PASS", path)
    else:
        monkeypatch.delenv("LBMC_PASS", raising=False)
    lats = [cases.build(lbmc.Lattice, c, storage=storage) for c in group]
    assert all((lat.pass_info()["calls"] == 1) == (path == "0") for lat in lats)
    assert sum(lat.n for lat in lats) >= 1 << 20
    model = None
    if every:
        model = lbmc.Mlp(pymlp.flatten(pymlp.init_params(3)), mu=[0] * 6 + [1], isd=[300.0] * 6 + [100.0], out_a=0.02,
                         out_b=0.8)
        for lat in lats[3:5]:
            lat.set_closure(model, 0.6, 1.0)
            lat.set_closure_interval(every)
    batch = lbmc.Batch(lats)
    for t0, n in runs:
        batch.run(t0, n, store_every)
    out = []
    for lat in lats:
        rho, u = lat.get_macros()
        out += [lat.get_f(), rho, u]
    batch.close()
    for lat in lats:
        lat.close()
    if model is not None:
        model.close()
    return out


@pytest.mark.parametrize("storage,every,store_every", [
    (0, 0, 4), (1, 0, 7), (1, 0, 0), (1, 1, 9), (1, 2, 1), (1, 3, 5), (1, 8, 9)])
def test_large_batches(monkeypatch, storage, every, store_every):
    # prescribed values where their calls are stored seldom enough
    group = _group(prescribed=store_every not in (1, 5))
    runs = [(3, 31), (34, 2), (36, 9)]
    want = _stepped(monkeypatch, "0", group, storage, every, store_every, runs)
    got = _stepped(monkeypatch, None, group, storage, every, store_every, runs)
    for k, (g, w) in enumerate(zip(got, want)):
        assert np.array_equal(g, w), k // 3
