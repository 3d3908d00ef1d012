"""Read-back and set_f through the pinned staging memory, exactly: against
the path with the library's fixed scratch, single-node reads and the values
written, at sizes around the limits between its ways of copying."""
import threading

import numpy as np
import pytest

import closure

pytestmark = pytest.mark.gpu
lbmc = pytest.importorskip("lbmc")

# rho and u (FP32): 60 bytes; 4 below and 8 above 1 MB; odd pieces; 60 MB
SIZES = [(5, 1), (29127, 3), (43691, 2), (1031, 613), (2503, 2011)]

W = np.array([4 / 9] + 4 * [1 / 9] + 4 * [1 / 36])[:, None]
NOALLOC = threading.Lock()  # one call at a time, as its description asks


def _noalloc(lat):
    with NOALLOC:
        return lat.get_f_noalloc()


def _lattice(length, storage, seed=0):
    n = length[0] * length[1]
    lat = lbmc.Lattice(lattice=lbmc.D2Q9, length=length, storage=storage, tau=0.8)
    lat.set_fields(geometry=np.zeros(n))
    rng = np.random.default_rng(seed)
    lat.init_equilibrium(1 + 0.01 * rng.standard_normal(n), 0.01 * rng.standard_normal((2, n)))
    f = _noalloc(lat)
    # every element its own value
    f = np.float32(f * (1 + 0.001 * rng.standard_normal(f.shape))).astype(np.float64)
    return lat, f


def _check(lat, f):
    lat.set_f(f)
    # FP32 populations are kept as their distance from the weights
    want = f if lat.storage == 0 else W + np.float32(f - W).astype(np.float64)
    assert np.array_equal(lat.get_f(), want)
    assert np.array_equal(_noalloc(lat), want)
    lat.run(0, 1, 1)
    rho, u = lat.get_macros()
    n = rho.size
    for k in {0, 1, n // 3, n // 2, n - 2, n - 1}:
        r, v = lat.get_node(k)
        assert r == rho[k] and np.array_equal(v, u[:, k])
    g = lat.get_f()  # the copy is ordered behind the run
    assert np.array_equal(g, _noalloc(lat))


@pytest.mark.parametrize("storage", [0, 1], ids=["f64", "f32"])
@pytest.mark.parametrize("length", SIZES, ids=lambda s: "%dx%d" % s)
def test_transfers_are_exact(length, storage):
    lat, f = _lattice(length, storage)
    _check(lat, f)
    lat.close()


def test_threads_transfer_at_once():
    lats = [_lattice((1031, 613), k % 2, k) for k in range(4)]
    errors = []

    def work(lat, f):
        try:
            for _ in range(3):
                _check(lat, f)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=lf) for lf in lats]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for lat, _ in lats:
        lat.close()


def test_forward_of_any_size_and_from_threads():
    rng = np.random.default_rng(3)
    x = np.float32(rng.standard_normal((3_000_001, 7)))
    m = lbmc.Mlp(closure.init_params(1))
    # parts of 256 samples, each through the smallest transfers
    want = np.concatenate([m.forward(x[k:k + 256]) for k in range(0, 200_000, 256)])[:200_000]
    for s in (1, 255, 74898, 74899, 200_000, 1_000_003, 3_000_001, 200_000):
        y = m.forward(x[:s])
        k = min(s, 200_000)
        assert y.shape == (s,) and np.array_equal(y[:k], want[:k])
    whole = m.forward(x)
    bad = []

    def work(s):
        for _ in range(3):
            if not np.array_equal(m.forward(x[-s:]), whole[-s:]):
                bad.append(s)

    threads = [threading.Thread(target=work, args=(256 * s,)) for s in (1, 300, 1000, 4000)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    m.close()
