"""Passes of several calls (lbmc_run) against one call per
launch, bit for bit: the same node updates in another order of memory traffic.
LBMC_PASS=0 keeps one call per launch; "size,W,H,M" (D2Q9) and "W,H,nz"
(D3Q15) force a tile shape."""
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


@pytest.mark.parametrize("storage", [1, 2], ids=["f32", "f16s"])
def test_planned_shape_between_pressure_faces(monkeypatch, storage):
    # large enough that the planner limits the tiles of a lattice with boundary nodes
    case = cases.pressure_d2q9(Lx=701, Ly=397, collision=cases.MRT)
    want = _run(monkeypatch, case, storage, "0", 5)
    got = _run(monkeypatch, case, storage, None, 5)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


def test_long_time_index_and_late_start(monkeypatch):
    case = cases.channel_d2q9(37, 21)
    want = _run(monkeypatch, case, 0, "0", 3, t0=2 ** 31 + 5)
    got = _run(monkeypatch, case, 0, None, 3, t0=2 ** 31 + 5)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


def _duct(forcing):
    """A box with solid walls on four sides and a solid block inside."""
    L = (37, 22, 11)
    c = cases.turbulence_d3q15(1, forcing=False)
    n = L[0] * L[1] * L[2]
    rng = np.random.default_rng(5)
    geo = np.zeros((L[2], L[1], L[0]))
    geo[0] = geo[-1] = 1
    geo[:, 0] = geo[:, -1] = 1
    geo[4:6, 8:12, 10:17] = 1
    force = [np.full(n, 1e-5), 1e-6 * rng.standard_normal(n), np.zeros(n)] if forcing else None
    return dict(c, name=f"duct_d3q15_g{int(forcing)}",
                desc=dict(c["desc"], length=L, forcing=forcing, c_smag=0.1 if forcing else 0.0),
                fields=dict(geometry=geo.reshape(-1), force=force),
                init=("equilibrium", 1 + 0.01 * rng.standard_normal(n), cases.random_velocity(rng, (L[2], L[1], L[0]), 0.02)))


D3_CASES = [
    cases.turbulence_d3q15(12),
    cases.turbulence_d3q15(35, c_smag=0.0),
    cases.turbulence_d3q15(13, forcing=True),
    _duct(False),
    _duct(True),
    cases.turbulence_d3q15(12, collision=cases.MRT),
    cases.faces_d3q15(),                              # boundary nodes: no passes either
]


@pytest.mark.parametrize("storage", [0, 1, 2], ids=["f64", "f32", "f16s"])
@pytest.mark.parametrize("case", D3_CASES, ids=lambda c: c["name"])
def test_march_matches_one_call_per_launch(monkeypatch, case, storage):
    for store_every in (0, 1, 5):
        want = _run(monkeypatch, case, storage, "0", store_every)
        # whole rows and several z ranges, small uneven tiles, the smallest
        # tile with single-plane ranges, a tile larger than the lattice
        for shape in ("37,13,3", "9,7,2", "3,3,64", "64,8,1"):
            got = _run(monkeypatch, case, storage, shape, store_every)
            for a, b in zip(got, want):
                assert np.array_equal(a, b), (shape, store_every)


def _forced(case, uniform, collision, quirks):
    n = len(case["fields"]["geometry"])
    force = [np.full(n, 2e-5), np.full(n, -1e-6), np.zeros(n)] if uniform else case["fields"]["force"]
    rates = cases.d3q15_rates(0.7) if collision == cases.MRT else None
    return dict(case, desc=dict(case["desc"], collision_type=collision, quirks=quirks, tau_mrt=rates),
                fields=dict(case["fields"], force=force))


@pytest.mark.parametrize("storage", [0, 1], ids=["f64", "f32"])
@pytest.mark.parametrize("quirks", [0, 3])
@pytest.mark.parametrize("force", ["none", "node", "uniform"])
@pytest.mark.parametrize("collision", [cases.BGK, cases.MRT], ids=["bgk", "mrt"])
def test_march_of_forced_ducts(monkeypatch, collision, force, quirks, storage):
    # every kernel of the march: collision, force, MRT matrix; walls inside
    case = _forced(_duct(force != "none"), force == "uniform", collision, quirks)
    want = _run(monkeypatch, case, storage, "0", 4)
    for shape in ("37,13,3", "9,7,2"):
        got = _run(monkeypatch, case, storage, shape, 4)
        for a, b in zip(got, want):
            assert np.array_equal(a, b), shape


@pytest.mark.parametrize("storage", [0, 1], ids=["f64", "f32"])
def test_march_planned_shape(monkeypatch, storage):
    # large enough for the planner to choose passes by itself
    case = cases.turbulence_d3q15(1)
    L = (131, 96, 75)
    n = L[0] * L[1] * L[2]
    rng = np.random.default_rng(8)
    case = dict(case, desc=dict(case["desc"], length=L), fields=dict(geometry=np.zeros(n)),
                init=("equilibrium", 1 + 0.01 * rng.standard_normal(n),
                      cases.random_velocity(rng, (L[2], L[1], L[0]), 0.02)))
    want = _run(monkeypatch, case, storage, "0", 5)
    got = _run(monkeypatch, case, storage, None, 5)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


def _batch(monkeypatch, pass_env, storage, every, store_every, runs, swap_in=False):
    """Uneven members (plain BGK, MRT with forcing, prescribed values and, when
    every > 0, learned-closure members) stepped as a batch."""
    if pass_env is None:
        monkeypatch.delenv("LBMC_PASS", raising=False)
    else:
        monkeypatch.setenv("LBMC_PASS", pass_env)
    group = [cases.channel_d2q9(37, 21, collision=cases.MRT, rates=cases.d2q9_rates(0.8)),
             cases.channel_d2q9(130, 66), cases.pressure_d2q9(), cases.porous_d2q9(L=40, collision=cases.NTPOR),
             cases.channel_d2q9(64, 48), cases.channel_d2q9(90, 31)]
    lats = [cases.build(lbmc.Lattice, c, storage=storage) for c in group]
    model = None
    if every:
        import pymlp
        model = lbmc.Mlp(pymlp.flatten(pymlp.init_params(3)), mu=[0] * 6 + [1], isd=[300.0] * 6 + [100.0], out_a=0.02,
                         out_b=0.8)
        for lat in lats[4:]:
            lat.set_closure(model, 0.6, 1.0)
            lat.set_closure_interval(every)
    b = lbmc.Batch(lats)
    for t0, n in runs:
        b.run(t0, n, store_every)
        lats[1].step(t0 + n, False)  # a member on its own between batch runs
        lats[1].step(t0 + n + 1, False)
    out = []
    for lat in lats:
        rho, u = lat.get_macros()
        out.append((lat.get_f(), rho, u))
    b.close()
    for lat in lats:
        lat.close()
    if model is not None:
        model.close()
    return out


@pytest.mark.parametrize("storage,every", [(0, 0), (1, 0), (1, 1), (1, 2), (1, 4), (1, 8)],
                         ids=["f64", "f32", "every1", "every2", "every4", "every8"])
def test_batch_passes_match_one_call_per_launch(monkeypatch, storage, every):
    runs = [(3, 41), (44, 1), (45, 18), (2 ** 31 + 7, 9)]
    for store_every in (0, 4, 9):
        want = _batch(monkeypatch, "0", storage, every, store_every, runs)
        got = _batch(monkeypatch, None, storage, every, store_every, runs)
        for k, (w, g) in enumerate(zip(want, got)):
            for a, b in zip(g, w):
                assert np.array_equal(a, b), (k, store_every)


def _closure_run(monkeypatch, shape, case, every, store_every, band):
    monkeypatch.setenv("LBMC_PASS", shape)
    import pymlp
    model = lbmc.Mlp(pymlp.flatten(pymlp.init_params(3)), mu=[0] * 6 + [1], isd=[300.0] * 6 + [100.0], out_a=0.02,
                     out_b=0.8)
    lat = cases.build(lbmc.Lattice, case, storage=1)
    lat.set_closure(model, *band)
    lat.set_closure_interval(every)
    lat.run(3, 23, store_every)   # starts between evaluations, without a record
    lat.run(26, 1, 1)
    lat.run(27, every, 0)         # at most one pair: run one by one
    lat.run(27 + every, 4 * every, 2)
    f = lat.get_f()
    lat.set_f(f)                  # the record goes with the state
    lat.run(2 ** 31 + 2, 17, store_every)
    rho, u = lat.get_macros()
    out = lat.get_f(), rho, u
    lat.close()
    model.close()
    return out


@pytest.mark.parametrize("every", [2, 3, 4, 7, 8])
@pytest.mark.parametrize("case", D3_CASES[:5], ids=lambda c: c["name"])
def test_closure_passes_match_one_call_per_launch(monkeypatch, case, every):
    # the band of the second leaves nodes outside: the record's NaN entries
    for store_every, band in ((0, (0.6, 1.0)), (5, (0.799, 0.802))):
        want = _closure_run(monkeypatch, "0", case, every, store_every, band)
        for shape in ("37,13,3", "9,7,2", "64,8,1"):
            got = _closure_run(monkeypatch, shape, case, every, store_every, band)
            for a, b in zip(got, want):
                assert np.array_equal(a, b), (shape, store_every)
