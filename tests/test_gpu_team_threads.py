"""GPU: minimizations of several contexts at once: more teams than the device has room for (those that
find none take the four-kernel slots), and batches among them. Every result is the one it has alone."""
import threading

import numpy as np
import pytest

from picgo_amd import abi, mech, synth

pytestmark = pytest.mark.gpu


def _net(fil, cyl, seed):
    p = synth.preset(1)
    p.seed, p.n_fil, p.n_cyl_min, p.n_cyl_max, p.n_linkers, p.n_motors = seed, fil, cyl, cyl, 4 * fil, 2 * fil
    p.box = max(108.0 * (cyl + 2) / 3 ** 0.5 + 200, 2000.0)
    return synth.Network(p)


@pytest.mark.parametrize("prec", [abi.MDN_PREC_FP64, abi.MDN_PREC_MIXED])
def test_results_are_those_alone(gpu, prec):
    p = abi.default_cg_params(precision=prec, energy_call_limit=40)
    work = []
    for k, (fil, cyl) in enumerate([(50, 10), (50, 10), (120, 12), (200, 10), (20, 6), (150, 12)]):
        net = _net(fil, cyl, 40 + k)
        g = gpu()
        g.upload(net.desc, net.coord)
        g.reset_neighbor_lists(net.coord)
        work.append(lambda g=g, x=net.coord: [g.minimize(p, x)[:2], g.last_team()])
    for b in range(2):
        nets = [synth.Network.config(3, index=4 * b + i) for i in range(4)]
        gs = []
        for n in nets:
            gs.append(gpu())
            gs[-1].upload(n.desc, n.coord)
            gs[-1].reset_neighbor_lists(n.coord)
        work.append(lambda gs=gs, nets=nets: [sum(([x, f] for x, f in zip(*mech.minimize_batched(gs, p, [n.coord for n in nets])[:2])), []),
                                              gs[0].last_team()])
    want = [w()[0] for w in work]
    bad, forms = [], [set() for _ in work]

    def run(k):
        for _ in range(12):
            got, team = work[k]()
            forms[k].add(team)
            if not all(np.array_equal(a, b) for a, b in zip(got, want[k])):
                bad.append((k, team))

    ts = [threading.Thread(target=run, args=(k,)) for k in range(len(work))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    print(forms, flush=True)
    assert not bad
    assert all(w()[1][0] > 0 for w in work)   # alone again: by teams, so the room was given back
