"""GPU: lists of clumped networks, where a cylinder has more neighbours than one search keeps (32) and a
tile's halo more members than LDS holds (512): the pairs and their order are the predicate's over every
pair of cylinders, also at the grid's corner, with clumps beside sparse filaments, and for a binder's
list; and a search takes milliseconds (by insertion sort with one lane in eight: a second)."""
import ctypes as C
import time

import numpy as np
import pytest

from picgo_amd import abi, mech, synth
from tests.test_gpu_neighbor_dense import _pairs

pytestmark = pytest.mark.gpu


def _made(fil, cyl, box, spread, seed=29):
    """Filaments thrown into a clump, every seventh left where it was."""
    p = synth.preset(0)
    p.n_fil, p.n_cyl_min, p.n_cyl_max, p.box, p.seed, p.n_linkers, p.n_motors = fil, cyl, cyl, box, seed, 0, 0
    net = synth.Network(p)
    X = net.coord.reshape(fil, cyl + 1, 3).copy()
    c = X.mean(1, keepdims=True)
    to = 260.0 + spread * np.random.default_rng(seed).random((fil, 1, 3))
    X = np.where((np.arange(fil) % 7 == 0)[:, None, None], X, X - c + to)
    x = np.clip(X, 1.0, box - 1.0).reshape(-1)
    g = mech.ForceFieldManager(0)
    g.upload(net.desc, x)
    return net, x, g


@pytest.mark.parametrize("fil,cyl,box,spread", [(40, 3, 2000.0, 120.0), (150, 4, 2000.0, 60.0), (420, 3, 3000.0, 200.0),
                                                (700, 2, 1400.0, 450.0)])
def test_clumps(fil, cyl, box, spread):
    net, x, g = _made(fil, cyl, box, spread)
    want = _pairs(net, x)
    assert np.bincount(want[:, 0]).max() > 32
    for _ in range(2):
        assert g.reset_neighbor_lists(x) == len(want) and np.array_equal(g.neighbor_pairs(), want)


def test_binding_list_of_a_dense_network():
    p = synth.preset(1)
    p.n_fil, p.n_cyl_min, p.n_cyl_max, p.seed, p.box = 600, 12, 12, 7, 1080.0
    p.n_linkers, p.n_motors = 2400, 1200
    net = synth.Network(p)
    x = net.coord + np.random.default_rng(1).normal(0, 2, net.coord.size)
    g = mech.ForceFieldManager(0)
    g.upload(net.desc, x)
    b = abi.binding_params(np.array([0.125, 0.375, 0.625, 0.875]), 30.0, 40.0, 108.0)
    n, room = C.c_int64(), 400 * net.n_cylinders
    out = np.zeros((room, 2), np.uint32)
    took, got = [], []
    for _ in range(3):
        t = time.perf_counter()
        st = mech.lib().mdn_binding_pairs(g._h, C.byref(b), x.ctypes.data_as(C.POINTER(C.c_double)),
                                          out.ctypes.data_as(C.POINTER(C.c_uint32)), room, C.byref(n))
        took.append(time.perf_counter() - t)
        assert st == 0
        got.append(out[:n.value].copy())
    print(f"{net.n_beads} beads: {n.value} sites in {min(took) * 1e3:.2f} ms", flush=True)
    assert n.value > 100000 and np.array_equal(got[0], got[1]) and np.array_equal(got[1], got[2])
    assert min(took) < 0.1
