"""GPU: results to the host at sizes around those where the way they are copied changes (256 KB, 768 KB
and 2 MB) and below, bit for bit, from an idle stream and behind queued kernels, into memory that is
mapped and into fresh pages, aligned to pages and not; and parameters uploaded one after another from
buffers that are overwritten as soon as the call returns."""
import ctypes
import mmap

import numpy as np
import pytest

from picgo_amd import autograd, mech, synth

pytestmark = pytest.mark.gpu


def _ctx(fil, cyl, wide=1.0):
    p = synth.preset(1)
    p.n_fil, p.n_cyl_min, p.n_cyl_max, p.seed = fil, cyl, cyl, 7
    p.box = wide * max(3000.0, 1000.0 * (fil * cyl / 95.0) ** (1 / 3))
    p.n_linkers = p.n_motors = 0
    net = synth.Network(p)
    g = mech.ForceFieldManager(0)
    g.upload(net.desc, net.coord)
    return net, g


def _get(g, a):
    st = mech.lib().mdn_get_coords(g._h, a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)))
    assert st == 0
    return a


SIZES = [32, 33, 195, 196, 520, 521, 1560, 1561, 4161, 4162]   # filaments of 21 beads, 504 bytes, each


@pytest.mark.parametrize("fil", SIZES)
def test_product_into_mapped_and_fresh_pages(fil):
    """Behind the product's kernels: H v, the same whatever memory receives it (in a wide box: a pair of
    crossing filaments may have no tangent)."""
    net, g = _ctx(fil, 20, 10.0)
    x = net.coord + np.random.default_rng(fil).normal(0.0, 1.0, net.coord.size)
    v = np.random.default_rng(1).normal(size=x.size)
    g.reset_neighbor_lists(x)
    p = [a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for a in (x, v)]
    want = None
    for at in (None, None, 0, 8):
        if at is None:
            a = np.full(x.size, 7.0)
        else:
            m = mmap.mmap(-1, x.nbytes + 8192)
            a = np.frombuffer(m, np.float64, x.size, at)
        assert mech.lib().mdn_hvp(g._h, *p, a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), x.size) == 0
        want = a.copy() if want is None else want
        assert want.any() and np.array_equal(a, want)


@pytest.mark.parametrize("fil", SIZES)
def test_result_into_mapped_and_fresh_pages(fil):
    net, g = _ctx(fil, 20)
    x = np.random.default_rng(fil).normal(500.0, 100.0, net.coord.size)
    for k in range(2):
        g.set_coords(x)
        mapped = np.full(x.size + 1, 7.0)
        assert np.array_equal(_get(g, mapped[1:]), x) and mapped[0] == 7.0
        for at in (0, 8):
            m = mmap.mmap(-1, x.nbytes + 8192)
            a = np.frombuffer(m, np.float64, x.size, at)
            assert np.array_equal(_get(g, a), x)
            assert not any(m[at + x.nbytes:]) and not any(m[:at])
            del a
        x = -x


@pytest.mark.parametrize("fil,cyl", [(50, 10), (600, 14)])   # 4 KB and 67 KB a parameter
def test_parameters_from_buffers_that_are_reused(fil, cyl):
    net, g = _ctx(fil, cyl)
    g.reset_neighbor_lists(net.coord)
    th = autograd.theta0(net.desc).numpy()
    one, two = th * 1.25, th * 0.875

    def install(t, spoil):
        buf = t.copy()
        st = mech.lib().mdn_set_params(g._h, *(r.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for r in buf))
        assert st == 0
        if spoil:
            buf[:] = -1e30

    install(one, False)
    e1, f1 = g.compute_energy(net.coord), g.compute_forces(net.coord)
    install(two, False)
    assert g.compute_energy(net.coord) != e1
    for k in range(5):
        install(one, True)
        assert g.compute_energy(net.coord) == e1 and np.array_equal(g.compute_forces(net.coord), f1)
