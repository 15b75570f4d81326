"""GPU: coordinates to the device and back through the pinned ring, bit for bit, at sizes below its
minimum, within one chunk, between the small and the large sizes that go through it, and beyond
the whole ring (5 MB through 4 MB); from memory that is not 16-byte aligned; and by more threads
than there are rings."""
import threading

import numpy as np
import pytest

from picgo_amd import mech, synth

pytestmark = pytest.mark.gpu


def _ctx(fil, cyl, seed):
    p = synth.preset(1)
    p.n_fil, p.n_cyl_min, p.n_cyl_max, p.seed = fil, cyl, cyl, 7
    p.box = max(3000.0, 1000.0 * (fil * cyl / 95.0) ** (1 / 3))
    p.n_linkers = p.n_motors = 0
    net = synth.Network(p)
    g = mech.ForceFieldManager(0)
    g.upload(net.desc, net.coord)
    return g, np.random.default_rng(seed).normal(500.0, 100.0, net.coord.size)


def _round(g, x):
    g.set_coords(x)
    assert np.array_equal(g.get_coords(), x)
    g.set_coords(x[::-1].copy())
    y = g.get_coords()
    assert np.array_equal(y, x[::-1])


@pytest.mark.parametrize("fil,cyl", [(2, 2), (7, 11), (900, 9), (2300, 9), (9000, 24)])
def test_round_trip(fil, cyl):
    g, x = _ctx(fil, cyl, fil)
    _round(g, x)
    off = np.empty(x.size + 1)[1:]   # memory that is not 16-byte aligned
    off[:] = x
    g.set_coords(off)
    assert np.array_equal(g.get_coords(), x)


def test_more_threads_than_rings():
    made = [_ctx(900 + k, 9, k) for k in range(6)]
    bad = []

    def work(g, x):
        for _ in range(20):
            g.set_coords(x)
            if not np.array_equal(g.get_coords(), x):
                bad.append(x.size)

    ts = [threading.Thread(target=work, args=m) for m in made]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
