"""GPU: the FP64 line search of dense networks, on both sides of the number of pairs beyond which a
pair's forces and energy stay in one thread: the forces a minimization returns are those of a force
evaluation at its coordinates, bit for bit."""
import numpy as np
import pytest

from picgo_amd import abi, mech, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box,pairs", [(3600.0, (140000, 190000)), (3200.0, (210000, 260000))])
def test_forces_are_those_of_an_evaluation(box, pairs):
    p = synth.preset(1)
    p.n_fil, p.n_cyl_min, p.n_cyl_max, p.box, p.seed = 2000, 20, 20, box, 7
    net = synth.Network(p)
    x = net.coord + np.random.default_rng(3).normal(0.0, 2.0, net.coord.size)
    g = mech.ForceFieldManager(0)
    g.upload(net.desc, x)
    n = g.reset_neighbor_lists(x)
    assert pairs[0] < n < pairs[1], n
    y, f, r = g.minimize(abi.default_cg_params(energy_call_limit=12), x)
    assert r.num_iter > 0 and np.array_equal(f, g.compute_forces(y))
