"""GPU: the persistent minimizer (teams of workgroups, one kernel per minimization).

Bars:
  a single network's result (coordinates, forces, counts, energies) is bit-identical for every team
    size and to the four-kernel slots, at sizes around a wavefront's 64 beads and a block's 256, in
    both precisions and with the beads renumbered;
  a batch's results are bit-identical for every number of workgroups, from one (each system pulled
    from the queue) to a team of several per system.
"""
import os

import numpy as np
import pytest

from picgo_amd import abi, mech, synth

pytestmark = pytest.mark.gpu


def _ctx(gpu, desc, x, size=None):
    if size is not None:
        os.environ["MDN_CG_TEAM"] = str(size)
    try:
        g = gpu()
    finally:
        os.environ.pop("MDN_CG_TEAM", None)
    g.upload(desc, x)
    g.reset_neighbor_lists(x)
    return g


def _same(a, b):
    (xa, fa, ra), (xb, fb, rb) = a, b
    np.testing.assert_array_equal(xa, xb)
    np.testing.assert_array_equal(fa, fb)
    assert (ra.num_iter, ra.num_energy_call, ra.num_force_call, ra.num_safe_mode) == \
        (rb.num_iter, rb.num_energy_call, rb.num_force_call, rb.num_safe_mode)
    assert ra.energies_after.total == rb.energies_after.total


@pytest.mark.parametrize("n_fil,n_cyl", [(1, 1), (9, 6), (8, 7), (13, 4), (16, 15), (40, 9)])
@pytest.mark.parametrize("prec", [abi.MDN_PREC_FP64, abi.MDN_PREC_MIXED])
def test_team_sizes_equal_the_slots(gpu, n_fil, n_cyl, prec):
    # 2, 63, 64, 65, 256 and 400 beads
    net = synth.Network.config(0, n_fil=n_fil, n_cyl_min=n_cyl, n_cyl_max=n_cyl, n_linkers=min(20, n_fil), seed=n_fil)
    x = net.coord + np.random.default_rng(n_fil).normal(0.0, 2.0, net.coord.size)
    p = abi.default_cg_params(precision=prec, energy_call_limit=60)
    ref = _ctx(gpu, net.desc, x, 0).minimize(p, x)
    for size in (None, 1, 2, 5, 16, 32):
        _same(_ctx(gpu, net.desc, x, size).minimize(p, x), ref)


def test_team_with_renumbered_beads_and_safe_mode(gpu):
    """A dense network (safe-mode entries, recovery moves, several halvings per search) with its
    beads renumbered: the neighbour tables, the second trial and the moves, in a team."""
    from tests.test_gpu_bonded_gather import _relabelled
    net = synth.Network.config(3, index=4, dense=True)
    d, x, _ = _relabelled(net.desc, net.coord, 5)
    p = abi.default_cg_params(energy_call_limit=60)
    ref = _ctx(gpu, d, x, 0).minimize(p, x)
    assert ref[2].num_safe_mode > 0
    for size in (3, 16):
        _same(_ctx(gpu, d, x, size).minimize(p, x), ref)


@pytest.mark.parametrize("prec", [abi.MDN_PREC_FP64, abi.MDN_PREC_MIXED])
def test_batch_results_do_not_depend_on_the_workgroups(gpu, prec):
    nets = [synth.Network.config(3, index=i, dense=i % 3 == 2) for i in range(9)]
    ffms = [_ctx(gpu, n.desc, n.coord) for n in nets]
    p = abi.default_cg_params(precision=prec, energy_call_limit=50)
    ref = None
    for cap in (None, 1, 7, 20, 100):
        if cap is not None:
            os.environ["MDN_BATCH_MAX_WORKGROUPS"] = str(cap)
        try:
            xs, fs, rs = mech.minimize_batched(ffms, p, [n.coord for n in nets])
        finally:
            os.environ.pop("MDN_BATCH_MAX_WORKGROUPS", None)
        if ref is None:
            ref = xs, fs, rs
        for i in range(len(nets)):
            _same((xs[i], fs[i], rs[i]), (ref[0][i], ref[1][i], ref[2][i]))
