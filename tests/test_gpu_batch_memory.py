"""GPU: a batch's coordinates and forces in ordinary, pinned and device memory, in one call: the same
bits wherever they are, as a single minimization takes them from all three."""
import ctypes as C

import numpy as np
import pytest
import torch

from picgo_amd import abi, mech, synth

pytestmark = pytest.mark.gpu

DP = C.POINTER(C.c_double)


def _buffers(x, where):
    """Coordinates x and room for forces, in memory of the kind asked for."""
    if where == "device":
        return torch.from_numpy(x).cuda(), torch.zeros(x.size, dtype=torch.float64, device="cuda")
    a = [torch.empty(x.size, dtype=torch.float64, pin_memory=where == "pinned") for _ in range(2)]
    a[0].copy_(torch.from_numpy(x))
    return a


def _made(k):
    nets = [synth.Network.config(3, index=i) for i in range(k)]
    ffms = []
    for n in nets:
        g = mech.ForceFieldManager(0)
        g.upload(n.desc, n.coord)
        g.reset_neighbor_lists(n.coord)
        ffms.append(g)
    return nets, ffms


def _ptr(t):
    return C.cast(t.data_ptr(), DP)


def test_batch_takes_coordinates_from_any_memory():
    nets, ffms = _made(6)
    p = abi.default_cg_params(energy_call_limit=40)
    want = mech.minimize_batched(ffms, p, [n.coord for n in nets])
    for kinds in (["pageable", "pinned", "device"] * 2, ["device"] * 6):
        bufs = [_buffers(n.coord, w) for n, w in zip(nets, kinds)]
        torch.cuda.synchronize()
        res = (abi.MinResult * 6)()
        st = mech.lib().mdn_minimize_batched((C.c_void_p * 6)(*[g._h.value for g in ffms]), 6, C.byref(p),
                                             (DP * 6)(*[_ptr(b[0]) for b in bufs]),
                                             (DP * 6)(*[_ptr(b[1]) for b in bufs]), res)
        assert st == 0
        for i, b in enumerate(bufs):
            assert np.array_equal(b[0].cpu().numpy(), want[0][i]), kinds[i]
            assert np.array_equal(b[1].cpu().numpy(), want[1][i]), kinds[i]
            assert res[i].num_iter == want[2][i].num_iter


@pytest.mark.parametrize("where", ["pageable", "pinned", "device"])
def test_single_minimization_does_too(where):
    nets, ffms = _made(1)
    p = abi.default_cg_params(energy_call_limit=40)
    x, f, _ = ffms[0].minimize(p, nets[0].coord)
    bx, bf = _buffers(nets[0].coord, where)
    torch.cuda.synchronize()
    res = abi.MinResult()
    assert mech.lib().mdn_minimize(ffms[0]._h, C.byref(p), _ptr(bx), _ptr(bf), C.byref(res)) == 0
    assert np.array_equal(bx.cpu().numpy(), x) and np.array_equal(bf.cpu().numpy(), f)
