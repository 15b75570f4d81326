"""GPU: the neighbor-list kernels where their paths change, against the list's predicate evaluated
over every pair of cylinders on the host: sparse bins, up to 32 neighbours of a cylinder (found and
ordered in LDS in one search), more (searched again and sorted in global memory), and halos with
more members than are staged in LDS (512). Pairs and their order are exact."""
import numpy as np
import pytest

from picgo_amd import mech, synth

pytestmark = pytest.mark.gpu


def _pairs(net, x):
    """Every pair in range, by the predicate (squares of the float ranges), in list order."""
    d = net.desc
    off = np.ctypeslib.as_array(d.fil_bead_offset, (d.n_filaments + 1,)).astype(int)
    beads = np.ctypeslib.as_array(d.fil_beads, (off[-1],)).astype(int)
    b1, b2, fil, pos = [], [], [], []
    for f in range(d.n_filaments):
        w = beads[off[f]:off[f + 1]]
        b1 += list(w[:-1]); b2 += list(w[1:])
        fil += [f] * (len(w) - 1); pos += list(range(len(w) - 1))
    X, fil, pos = x.reshape(-1, 3), np.array(fil), np.array(pos)
    mid = 0.5 * (X[b1] + X[b2])
    hi, lo = np.float64(np.float32(d.exvol_rmax) ** 2), np.float64(np.float32(d.exvol_rmin) ** 2)
    out = []
    for c in range(len(mid)):
        d2 = ((mid[:c] - mid[c]) ** 2).sum(1)
        keep = ~((d2 < lo) | (d2 > hi)) & ~((fil[:c] == fil[c]) & (abs(pos[:c] - pos[c]) <= 2))
        cn = np.nonzero(keep)[0]
        out.append(np.stack([np.full(len(cn), c), cn], 1))
    return np.concatenate(out)


# filaments x cylinders, box: a few filaments in a wide box; the ordinary density; clumps in one
# corner of a wide box, with up to 32, and with more than 32 neighbours and 512 cylinders near one bin
@pytest.mark.parametrize("fil,cyl,box,shrink", [(4, 3, 3000.0, 1.0), (50, 10, 2000.0, 1.0), (130, 6, 2000.0, 0.4),
                                                (300, 6, 2000.0, 0.3)])
def test_list_is_the_predicates(fil, cyl, box, shrink):
    p = synth.preset(0)
    p.n_fil, p.n_cyl_min, p.n_cyl_max, p.box, p.seed = fil, cyl, cyl, box, 17
    net = synth.Network(p)
    x = net.coord + np.random.default_rng(5).normal(0.0, 2.0, net.coord.size)
    if shrink < 1.0:   # filaments moved towards a corner, their shapes kept
        X, nb = x.reshape(fil, cyl + 1, 3), 300.0
        c = X.mean(1, keepdims=True)
        x = (X - c + nb + shrink * (c - nb)).reshape(-1).clip(1.0, box - 1.0)
    g = mech.ForceFieldManager(0)
    g.upload(net.desc, x)
    n = g.reset_neighbor_lists(x)
    want = _pairs(net, x)
    got = g.neighbor_pairs()
    most = np.bincount(want[:, 0]).max() if len(want) else 0
    assert (shrink > 0.35) == (most <= 32)
    assert n == len(want) and np.array_equal(got, want)
    assert g.reset_neighbor_lists(x) == n and np.array_equal(g.neighbor_pairs(), got)
