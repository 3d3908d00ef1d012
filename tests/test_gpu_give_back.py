"""The second population buffers of lattices that run in passes, given back
when an allocation of the library finds no memory (LBMC_OOM=n: none for n bytes
or more until a buffer was given back): the state stays, and the runs that
follow go one call per launch, with the same bits."""
import threading

import numpy as np
import pytest

import cases
import pymlp

pytestmark = pytest.mark.gpu
lbmc = pytest.importorskip("lbmc")


def _calls(lat):
    return lat.pass_info()["calls"]


def _read(lat):
    rho, u = lat.get_macros()
    return lat.get_f_noalloc(), rho, u


def _alone(monkeypatch, case, storage, calls):
    monkeypatch.setenv("LBMC_PASS", "0")
    lat = cases.build(lbmc.Lattice, case, storage=storage)
    monkeypatch.delenv("LBMC_PASS")
    assert _calls(lat) == 1
    lat.run(0, calls, 3)
    out = _read(lat)
    lat.close()
    return out


def _same(got, want):
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("storage", [0, 1], ids=["f64", "f32"])
def test_given_back_to_another_lattice(monkeypatch, storage):
    case = cases.channel_d2q9(301, 203)
    want = _alone(monkeypatch, case, storage, 90)
    lats = [cases.build(lbmc.Lattice, case, storage=storage) for _ in range(2)]
    other = cases.build(lbmc.Lattice, cases.channel_d2q9(64, 48), storage=1)
    assert all(_calls(lat) > 1 for lat in (*lats, other))
    for lat in lats:
        lat.run(0, 41, 3)  # not waited for
    monkeypatch.setenv("LBMC_OOM", "1")
    other.get_f()
    monkeypatch.delenv("LBMC_OOM")
    assert [_calls(lat) for lat in (*lats, other)] == [1, 1, 1]
    for lat in lats:
        lat.run(41, 49, 3)
        _same(_read(lat), want)
    lats[0].set_fields(**case["fields"])  # planned again
    assert _calls(lats[0]) > 1
    for lat in (*lats, other):
        lat.close()


def test_nothing_to_give_back(monkeypatch):
    lat = cases.build(lbmc.Lattice, cases.sf_d2q9(), storage=1)
    f = lat.get_f()
    monkeypatch.setenv("LBMC_OOM", "1")
    with pytest.raises(lbmc.LbmcError):
        lat.get_f()
    monkeypatch.delenv("LBMC_OOM")
    _same((lat.get_f(),), (f,))
    lat.close()


def test_batch_without_memory_for_its_lists(monkeypatch):
    # the only closure member drops its closure: the tile lists are built anew
    group = [cases.channel_d2q9(90, 31), cases.channel_d2q9(130, 66)]
    model = lbmc.Mlp(pymlp.flatten(pymlp.init_params(3)), mu=[0] * 6 + [1], isd=[300.0] * 6 + [100.0], out_a=0.02,
                     out_b=0.8)
    want = [_alone(monkeypatch, c, 1, 30) for c in group]
    lats = [cases.build(lbmc.Lattice, c, storage=1) for c in group]
    lats[0].set_closure(model, 0.6, 1.0)
    batch = lbmc.Batch(lats)
    lats[0].set_closure(None)
    monkeypatch.setenv("LBMC_OOM", "1")
    batch.run(0, 30, 3)
    monkeypatch.delenv("LBMC_OOM")
    assert [_calls(lat) for lat in lats] == [1, 1]
    for lat, w in zip(lats, want):
        _same(_read(lat), w)
    batch.close()
    for lat in lats:
        lat.close()
    model.close()


def test_given_back_while_others_run(monkeypatch):
    case = cases.channel_d2q9(301, 203)
    want = _alone(monkeypatch, case, 1, 200)
    lats = [cases.build(lbmc.Lattice, case, storage=1) for _ in range(3)]
    other = cases.build(lbmc.Lattice, cases.sf_d2q9(), storage=1)
    errors, busy = [], threading.Event()

    def work(lat):
        try:
            for t in range(0, 200, 20):
                lat.run(t, 20, 3)
                lat.sync()
                busy.set()
            lat.sync()
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(lat,)) for lat in lats]
    monkeypatch.setenv("LBMC_OOM", "1")
    for t in threads:
        t.start()
    busy.wait()
    try:
        other.get_f()
    except lbmc.LbmcError:
        pass  # every buffer was in use
    for t in threads:
        t.join()
    monkeypatch.delenv("LBMC_OOM")
    assert not errors
    for lat in lats:
        _same(_read(lat), want)
        lat.close()
    other.close()


def test_given_back_while_a_graph_is_captured(monkeypatch):
    # a closure lattice holds a buffer (for batches) and replays one call per
    # launch from a captured graph, 2016 launches long here
    case = cases.channel_d2q9(63, 32)
    model = lbmc.Mlp(pymlp.flatten(pymlp.init_params(3)), mu=[0] * 6 + [1], isd=[300.0] * 6 + [100.0], out_a=0.02,
                     out_b=0.8)

    def built():
        lat = cases.build(lbmc.Lattice, case, storage=1)
        lat.set_closure(model, 0.6, 1.0)
        return lat

    plain = built()
    for t in range(0, 4032, 7):
        plain.run(t, 7, 0)
    want = _read(plain)
    plain.close()
    other = cases.build(lbmc.Lattice, cases.sf_d2q9(), storage=1)
    for _ in range(4):
        lat, errors, begun, over = built(), [], threading.Event(), threading.Event()
        assert _calls(lat) > 1

        def work():
            begun.set()
            try:
                lat.run(0, 4032, 0)
            except BaseException as e:  # noqa: BLE001
                errors.append(e)
            over.set()

        monkeypatch.setenv("LBMC_OOM", "1")
        thread = threading.Thread(target=work)
        thread.start()
        begun.wait()
        while not over.is_set():
            try:
                other.get_f()
            except lbmc.LbmcError:
                pass  # the buffer was in use, or was given back before
        thread.join()
        monkeypatch.delenv("LBMC_OOM")
        assert not errors
        _same(_read(lat), want)
        lat.close()
    other.close()
    model.close()


def test_given_back_to_the_copy_measurement(monkeypatch):
    lat = cases.build(lbmc.Lattice, cases.channel_d2q9(64, 48), storage=1)
    small = cases.build(lbmc.Lattice, cases.channel_d2q9(32, 16), storage=1)
    # 1 MB each: the first finds a buffer to give back
    monkeypatch.setenv("LBMC_OOM", str(1 << 20))
    with pytest.raises(lbmc.LbmcError):
        lbmc.copy_bandwidth(1 << 20, 1)  # nothing left for the second
    monkeypatch.delenv("LBMC_OOM")
    assert _calls(lat) == _calls(small) == 1
    assert lbmc.copy_bandwidth(1 << 20, 1) > 0
    lat.close()
    small.close()


def test_training_after_a_step_without_memory(monkeypatch):
    rng = np.random.default_rng(4)
    x, y = np.float32(rng.standard_normal((20000, 7))), np.float32(rng.standard_normal(20000))
    out = []
    for fails in (False, True):
        model = lbmc.Mlp(pymlp.flatten(pymlp.init_params(3)))
        model.set_data(x, y)
        loss = [model.train(1, batch=64, seed=1)]
        if fails:
            monkeypatch.setenv("LBMC_OOM", "1")
            with pytest.raises(lbmc.LbmcError):
                model.train(1, batch=20000, seed=2)  # needs more gradient records
            monkeypatch.delenv("LBMC_OOM")
        loss.append(model.train(1, batch=64, seed=3))
        loss.append(model.train(1, batch=20000, seed=4))
        out.append([*loss, model.get_params()])
        model.close()
    _same(out[1], out[0])


def test_fields_without_memory_are_not_run(monkeypatch):
    case = cases.porous_d2q9(L=40, collision=cases.NTPOR)
    want = _alone(monkeypatch, case, 1, 20)
    lat = cases.build(lbmc.Lattice, case, storage=1)
    fields = case["fields"]
    # fluid everywhere: no buffer to give back, no porosity array yet
    monkeypatch.setenv("LBMC_PASS", "0")
    lat.set_fields(geometry=np.zeros(lat.n), force=fields["force"])
    monkeypatch.setenv("LBMC_OOM", "1")
    with pytest.raises(lbmc.LbmcError):
        lat.set_fields(**fields)
    monkeypatch.delenv("LBMC_OOM")
    for call in (lambda: lat.run(0, 5, 1), lambda: lat.step(0), lambda: lbmc.Batch([lat])):
        with pytest.raises(lbmc.LbmcError) as e:
            call()
        assert e.value.status == 4  # no fields
    lat.set_fields(**fields)
    lat.run(0, 20, 3)
    _same(_read(lat), want)
    lat.close()
