"""GPU: beads without filaments: a network with no interactions at all, through every minimizer (a zero
tolerance lets the line search run). There is no step to take, and every form says so."""
import numpy as np
import pytest

from picgo_amd import abi, mech
from tests.hand_systems import HandSystem

pytestmark = pytest.mark.gpu


def _system(n):
    hs = HandSystem([[np.array([100.0 + 5 * k, 500.0, 500.0]) for k in range(n)]], [])
    hs.desc.n_filaments = 0
    return hs


@pytest.mark.parametrize("n", [2, 70, 1100])
@pytest.mark.parametrize("prec", [abi.MDN_PREC_FP64, abi.MDN_PREC_MIXED])
def test_no_step_to_take(gpu, monkeypatch, n, prec):
    hs = _system(n)
    p = abi.default_cg_params(precision=prec, energy_call_limit=5)
    p.grad_tol = p.energy_rel_tol = 0.0
    for team in (0, 1, 3, "batch"):
        monkeypatch.setenv("MDN_CG_TEAM", "0" if team == "batch" else str(team))
        g = gpu()
        g.upload(hs.desc, hs.coord)
        assert g.reset_neighbor_lists(hs.coord) == 0
        with pytest.raises(mech.MdnError) as e:
            if team == "batch":
                mech.minimize_batched([g], p, [hs.coord])
            else:
                g.minimize(p, hs.coord)
        print(team, e.value, flush=True)
        assert e.value.code == 7   # MDN_ERR_RECOVERY
        assert not g.compute_forces(hs.coord).any() and g.compute_energy(hs.coord) == 0.0
