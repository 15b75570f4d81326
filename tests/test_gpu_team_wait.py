"""GPU: a team whose workgroups cannot all run. Its first barrier gives up after a bounded number of
polls, every workgroup ends, and the host minimizes without a team from the same start. Here the
bound is -1, at which everyone gives up, or zero polls, at which some may pass (and give up at the next
barrier, which sees that the others did). And teams of the sizes that
networks of some thousand beads get, on one XCD and spread over all of them (fences at every barrier).
Every result is the one without teams, bit for bit."""
import numpy as np
import pytest

from picgo_amd import abi, mech, synth
from tests.hand_systems import HandSystem

pytestmark = pytest.mark.gpu


def _made(gpu, monkeypatch, desc, x, **env):
    for k in ("MDN_CG_TEAM", "MDN_TEAM_POLLS", "MDN_TEAM_STRIDE"):
        if k in env:
            monkeypatch.setenv(k, str(env[k]))
        else:
            monkeypatch.delenv(k, raising=False)
    g = gpu()
    g.upload(desc, x)
    g.reset_neighbor_lists(x)
    return g


def _minimize(g, p, x, resident=False):
    if resident:
        g.set_coords(x)
        _, f, r = g.minimize(p, None)
        x = g.get_coords()
    else:
        x, f, r = g.minimize(p, x)
    return x, f, (r.num_iter, r.num_energy_call, r.num_force_call, r.num_safe_mode, r.energies_before.total,
                  r.energies_after.total, r.energy_rel_change)


def _same(a, b):
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and a[2] == b[2]


def _sphere(fil, cyl):
    n = fil * cyl
    r = max(500 + 54.0 * (cyl + 2), 10000.0 * (n / 400000) ** (1 / 3))
    p = synth.preset(4, radius=r, box=2 * r)
    p.seed, p.n_fil, p.n_cyl_min, p.n_cyl_max, p.n_linkers, p.n_motors = 11, fil, cyl, cyl, 4 * fil, 2 * fil
    net = synth.Network(p)
    return net, net.coord + np.random.default_rng(2).normal(0.0, 2.0, net.coord.size)


@pytest.mark.parametrize("team", [2, 16, 24])
@pytest.mark.parametrize("prec", [abi.MDN_PREC_FP64, abi.MDN_PREC_MIXED])
def test_single_network_whose_team_gives_up(gpu, monkeypatch, team, prec):
    net = synth.Network.config(0)
    x = net.coord + np.random.default_rng(1).normal(0.0, 2.0, net.coord.size)
    p = abi.default_cg_params(precision=prec, energy_call_limit=40)
    want = _minimize(_made(gpu, monkeypatch, net.desc, x, MDN_CG_TEAM=0), p, x)
    for polls in (-1, 0):
        g = _made(gpu, monkeypatch, net.desc, x, MDN_CG_TEAM=team, MDN_TEAM_POLLS=polls)
        for resident in (False, True, True, False):
            _same(_minimize(g, p, x, resident), want)
            assert g.last_team() == (0, 1) or (polls == 0 and g.last_team() == (team, 0))
    g = _made(gpu, monkeypatch, net.desc, x, MDN_CG_TEAM=team)   # and one that does not
    _same(_minimize(g, p, x), want)
    assert g.last_team() == (team, 0)


def test_forceN_pair_whose_team_gives_up(gpu, monkeypatch):
    a = np.array([500.0, 500.0, 500.0])
    hs = HandSystem([[a, a + [60.0, 0, 0]], [a + [80.0, 0, 0], a + [140.0, 0, 0]]], [])
    p = abi.default_cg_params(energy_call_limit=8)
    want = _minimize(_made(gpu, monkeypatch, hs.desc, hs.coord, MDN_CG_TEAM=0), p, hs.coord)
    g = _made(gpu, monkeypatch, hs.desc, hs.coord, MDN_CG_TEAM=3, MDN_TEAM_POLLS=-1)
    for _ in range(2):
        _same(_minimize(g, p, hs.coord), want)
        assert g.last_team() == (0, 1) and g.last_min_stats()["forceN_steps"] > 0


@pytest.mark.parametrize("prec", [abi.MDN_PREC_FP64, abi.MDN_PREC_MIXED])
def test_batch_whose_teams_give_up(gpu, monkeypatch, prec):
    nets = [synth.Network.config(3, index=i, dense=i == 4) for i in range(7)]
    p = abi.default_cg_params(precision=prec, energy_call_limit=40)

    def batch(given, **env):
        gs = [_made(gpu, monkeypatch, n.desc, n.coord, **env) for n in nets]
        x = [n.coord if given(i) else None for i, n in enumerate(nets)]
        xs, fs, rs = mech.minimize_batched(gs, p, x)
        xs = [g.get_coords() if y is None else y for g, y in zip(gs, xs)]
        return [(y, f, (r.num_iter, r.num_energy_call, r.energies_before.total, r.energies_after.total))
                for y, f, r in zip(xs, fs, rs)], gs[0].last_team()

    want, team = batch(lambda i: True)
    assert team[0] > 0 and team[1] == 0
    for given, polls in ((lambda i: True, -1), (lambda i: False, -1), (lambda i: i % 2, -1), (lambda i: i % 2, 0)):
        got, team = batch(given, MDN_TEAM_POLLS=polls)
        assert team[0] > 0 and (team[1] > 0 or polls == 0)
        for a, b in zip(got, want):
            _same(a, b)


def test_batch_with_a_failing_system_whose_teams_give_up(gpu, monkeypatch):
    """The status is still the failing system's, and the others are still returned."""
    a = np.array([500.0, 500.0, 500.0])
    hs = HandSystem([[a, a + [60.0, 0, 0]], [a + [80.0, 0, 0], a + [140.0, 0, 0]]], [])
    net = synth.Network.config(3, index=0)
    p = abi.default_cg_params(energy_call_limit=40)
    ref = mech.minimize_batched([_made(gpu, monkeypatch, net.desc, net.coord)], p, [net.coord])
    gs = [_made(gpu, monkeypatch, d.desc, d.coord, MDN_TEAM_POLLS=-1) for d in (net, hs)]
    with pytest.raises(mech.MdnError) as e:
        mech.minimize_batched(gs, p, [None, None])
    assert e.value.code == abi.MDN_ERR_UNSUPPORTED and "numerical force fallback" in str(e.value)
    assert gs[0].last_team()[1] == 1
    assert np.array_equal(gs[0].get_coords(), ref[0][0])


@pytest.mark.parametrize("fil,cyl", [(200, 20), (350, 20)])   # 4,200 and 7,350 beads
@pytest.mark.parametrize("prec", [abi.MDN_PREC_FP64, abi.MDN_PREC_MIXED])
def test_sizes_that_networks_get(gpu, monkeypatch, fil, cyl, prec):
    net, x = _sphere(fil, cyl)
    p = abi.default_cg_params(precision=prec, energy_call_limit=40)
    want = _minimize(_made(gpu, monkeypatch, net.desc, x, MDN_CG_TEAM=0), p, x)
    for env, team in (({}, None), (dict(MDN_CG_TEAM=24), 24), (dict(MDN_CG_TEAM=32), 32),
                      (dict(MDN_CG_TEAM=5, MDN_TEAM_STRIDE=1), 5), (dict(MDN_CG_TEAM=24, MDN_TEAM_STRIDE=1), 24)):
        g = _made(gpu, monkeypatch, net.desc, x, **env)
        _same(_minimize(g, p, x), want)
        assert g.last_team()[0] in ((16, 24) if team is None else (team,)) and g.last_team()[1] == 0, env
