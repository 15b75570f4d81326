"""GPU: the Simpson fallbacks in the persistent minimizer's teams. A team evaluates deferred pair
energies (energyN) by one workgroup of 512 threads while the others wait, the four-kernel slots by a
block of 1024; a step that needs the numerical forces (forceN) ends the kernel, and the host resumes
it. The result is the slots' bit for bit for every team size: the samples are summed in one order."""
import numpy as np
import pytest

from picgo_amd import abi
from tests.hand_systems import HandSystem

pytestmark = pytest.mark.gpu


def _pair(length, shift, gap, line):
    """Two parallel cylinders at a distance, or on one line with a gap, at their rest lengths: the
    pair's energy is the network's."""
    a = np.array([500.0, 500.0, 500.0])
    b = a + [length, 0, 0]
    c = (b + [gap, 0, 0]) if line else a + [shift, gap, 0]
    hs = HandSystem([[a, b], [c, c + [length - 7.0, 0, 0]]], [])
    hs._keep[4][:] = length, length - 7.0
    return hs


def _run(gpu, monkeypatch, hs, team, prec, calls):
    monkeypatch.setenv("MDN_CG_TEAM", str(team))
    g = gpu()
    g.upload(hs.desc, hs.coord)
    assert g.reset_neighbor_lists(hs.coord) == 1
    x, f, r = g.minimize(abi.default_cg_params(precision=prec, energy_call_limit=calls), hs.coord)
    return x, f, (r.num_iter, r.num_energy_call, r.num_force_call, r.energy_rel_change, r.grad_inf_norm,
                  r.energies_after.total), g.last_min_stats()["forceN_steps"]


@pytest.mark.parametrize("pair", [(81.0, 13.0, 31.0), (97.0, 5.0, 27.5), (66.0, 21.0, 38.0), (108.0, 0.0, 30.0)])
@pytest.mark.parametrize("prec", [abi.MDN_PREC_FP64, abi.MDN_PREC_MIXED])
def test_parallel_pair_is_the_slots(gpu, monkeypatch, pair, prec):
    hs = _pair(*pair, line=False)
    for calls in (1, 6):
        want = _run(gpu, monkeypatch, hs, 0, prec, calls)
        for team in (1, 3, 16):
            got = _run(gpu, monkeypatch, hs, team, prec, calls)
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]) and got[2] == want[2], team


@pytest.mark.parametrize("pair", [(60.0, 0.0, 20.0), (71.0, 0.0, 14.0), (66.0, 0.0, 9.0), (83.0, 0.0, 5.5)])
@pytest.mark.parametrize("prec", [abi.MDN_PREC_FP64, abi.MDN_PREC_MIXED])
def test_collinear_pair_is_the_slots(gpu, monkeypatch, pair, prec):
    hs = _pair(*pair, line=True)
    want = _run(gpu, monkeypatch, hs, 0, prec, 12)
    assert want[3] > 0
    for team in (1, 3, 16):
        got = _run(gpu, monkeypatch, hs, team, prec, 12)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]) and got[2:] == want[2:], team
