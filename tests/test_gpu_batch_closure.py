"""Members whose closure is switched on or off after lbmc_batch_create:
the batch reads the members' state at every run, so each member ends where
the same lattice stepped on its own ends, bit for bit."""
import numpy as np
import pytest

import cases
import pymlp

pytestmark = pytest.mark.gpu
lbmc = pytest.importorskip("lbmc")

GROUP = [cases.channel_d2q9(90, 31), cases.channel_d2q9(64, 48), cases.channel_d2q9(37, 21),
         cases.channel_d2q9(130, 66, collision=cases.MRT, rates=cases.d2q9_rates(0.8))]


def _model(seed):
    return lbmc.Mlp(pymlp.flatten(pymlp.init_params(seed)), mu=[0] * 6 + [1], isd=[300.0] * 6 + [100.0],
                    out_a=0.02, out_b=0.8)


def _read(lats):
    out = []
    for lat in lats:
        rho, u = lat.get_macros()
        out += [lat.get_f(), rho, u]
    return out


def _stepped(storage, on, phases, batched):
    """Closure members `on` = {member: interval} at first; phases: (changes
    {member: interval, or None for off}, calls)."""
    model = _model(3)
    lats = [cases.build(lbmc.Lattice, c, storage=storage) for c in GROUP]

    def switch(changes):
        for k, every in changes.items():
            lats[k].set_closure(model if every else None, 0.6, 1.0)
            if every:
                lats[k].set_closure_interval(every)

    switch(on)
    batch = lbmc.Batch(lats) if batched else None
    out, t = [], 3
    for changes, calls in phases:
        switch(changes)
        if batched:
            batch.run(t, calls, 5)
        else:
            for lat in lats:
                lat.run(t, calls, 5)
        t += calls
        out += _read(lats)
    if batched:
        batch.close()
    for lat in lats:
        lat.close()
    model.close()
    return out


@pytest.mark.parametrize("every", [1, 4])
@pytest.mark.parametrize("path", [None, "0"], ids=["passes", "one_call"])
@pytest.mark.parametrize("storage", [1, 2], ids=["f32", "f16s"])
def test_closure_switched_between_runs(monkeypatch, storage, path, every):
    if path is None:
        monkeypatch.delenv("LBMC_PASS", raising=False)
    else:
        monkeypatch.setenv("LBMC_PASS", path)
    # 75 calls: the captured graph of the one-call path, before and after a
    # change; up to 8: passes; one member off, another on, all off, the first
    # two on again
    phases = [({}, 75), ({}, 8), ({1: None, 2: every}, 8), ({}, 75), ({0: None, 2: None}, 7), ({}, 11),
              ({0: every, 1: every}, 8), ({}, 9)]
    want = _stepped(storage, {0: every, 1: every}, phases, False)
    got = _stepped(storage, {0: every, 1: every}, phases, True)
    for k, (g, w) in enumerate(zip(got, want)):
        assert np.array_equal(g, w), (k // (3 * len(GROUP)), k // 3 % len(GROUP))


@pytest.mark.parametrize("every", [1, 4])
def test_dropped_member_makes_each_call_once(every):
    # runs of even and odd numbers of passes: its state ends in either buffer
    phases = [({}, 9), ({1: None}, 21)] + [({}, n) for n in range(1, 13)]
    want = _stepped(1, {0: every, 1: every}, phases, False)
    got = _stepped(1, {0: every, 1: every}, phases, True)
    for k, (g, w) in enumerate(zip(got, want)):
        assert np.array_equal(g, w), (k // (3 * len(GROUP)), k // 3 % len(GROUP))


def test_dropped_member_without_a_record():
    """The member that drops its closure never had an interval above 1, so it
    holds no tau record; the others evaluate every 4th call and keep one."""
    phases = [({}, 9), ({1: None}, 21)]
    want = _stepped(1, {0: 4, 1: 1}, phases, False)
    got = _stepped(1, {0: 4, 1: 1}, phases, True)
    for g, w in zip(got, want):
        assert np.array_equal(g, w)


def test_weights_are_those_of_a_closure_member():
    """A member that took another model and then dropped the closure does not
    lend its weights to those that still have the batch's model."""
    first, other = _model(3), _model(11)
    out = []
    for batched in (False, True):
        lats = [cases.build(lbmc.Lattice, c, storage=1) for c in GROUP]
        for k in (0, 1):
            lats[k].set_closure(first, 0.6, 1.0)
        batch = lbmc.Batch(lats)
        lats[1].set_closure(other, 0.6, 1.0)
        with pytest.raises(lbmc.LbmcError) as e:
            batch.run(0, 4, 0)  # two models: refused
        assert e.value.status == 5
        lats[1].set_closure(None)
        if batched:
            batch.run(0, 40, 5)
        else:
            for lat in lats:
                lat.run(0, 40, 5)
        out.append(_read(lats))
        batch.close()
        for lat in lats:
            lat.close()
    first.close()
    other.close()
    for g, w in zip(out[1], out[0]):
        assert np.array_equal(g, w)
