"""lbmc_batch_autotune where runs go in passes: the shape it keeps is one of
the one-call launches, and it is what those are fastest with."""
import numpy as np
import pytest

import cases
import pymlp

pytestmark = pytest.mark.gpu
lbmc = pytest.importorskip("lbmc")


def test_autotune_times_the_launches_it_shapes():
    # members of 3072 nodes: chunks of 512, 1024 and 2048 nodes take 1.3, 1.8
    # and 2.7 times as long per call as chunks of 256
    lats = [cases.build(lbmc.Lattice, cases.channel_d2q9(64, 48), storage=1) for _ in range(16)]
    assert all(lat.pass_info()["calls"] > 1 for lat in lats)
    batch = lbmc.Batch(lats)
    shapes = []
    for k in range(6):
        grid, ms = batch.autotune(0, steps_per_trial=64)
        assert ms > 0 and batch.shape()[0] == grid
        shapes.append(batch.shape()[1])
    assert shapes == [256] * 6
    batch.close()
    for lat in lats:
        lat.close()


@pytest.mark.parametrize("storage,every", [(1, 1), (1, 4), (2, 4)])
def test_runs_after_autotune(monkeypatch, storage, every):
    # the closure members' chunks differ from the others' afterwards: bits of
    # the same lattices on their own, in passes and one call per launch
    group = [cases.channel_d2q9(90, 31), cases.channel_d2q9(300, 70), cases.pressure_d2q9()]
    model = lbmc.Mlp(pymlp.flatten(pymlp.init_params(3)), mu=[0] * 6 + [1], isd=[300.0] * 6 + [100.0], out_a=0.02,
                     out_b=0.8)

    def built():
        lats = [cases.build(lbmc.Lattice, c, storage=storage) for c in group]
        for lat in lats[:2]:
            lat.set_closure(model, 0.6, 1.0)
            lat.set_closure_interval(every)
        return lats

    alone = built()
    start = [lat.get_f() for lat in alone]
    lats = built()
    batch = lbmc.Batch(lats)
    for shape in (None, (1 << 20, 1024, 0), (5, 512, 0)):
        if shape is None:
            batch.autotune(0, steps_per_trial=5)
        else:
            batch.set_shape(*shape)
        for store_every in (8, 2):  # 2 with prescribed values: one call per launch
            for lat, one, f in zip(lats, alone, start):
                lat.set_f(f)
                one.set_f(f)
            batch.run(3, 70, store_every)
            for lat, one in zip(lats, alone):
                one.run(3, 70, store_every)
                assert np.array_equal(lat.get_f(), one.get_f())
    batch.close()
    for lat in (*lats, *alone):
        lat.close()
    model.close()
