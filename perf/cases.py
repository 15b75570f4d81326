"""Timed cases of the framework's own work, through its public entry points.

What a program that equilibrates actin networks has this library do, over the sizes that it meets:
one network between two chemistry steps (neighbor lists rebuilt, then a minimization), many
networks at once, single force evaluations from and into device memory, the lists that the
chemistry reads, and the derivatives that a parameter fit takes. A case is a dict of

    kind     which of those calls (the keys of RUNS)
    net      the network's shape: "cube" (six planes), "sphere" (one element), "replicas" (a batch)
    fil      filaments (of one network, or networks in a batch for "replicas")
    cyl      cylinders per filament, at most; at least `cyl_min`
    prec     "fp64" or "mixed"
    calls    the minimizer's energy-call limit (minimizations only)
    vecs     tangents of a Hessian-vector product (products only)

Networks come from the seeded generator at the densities of its presets, displaced by 2 nm of bead
noise, with crossing filaments pushed apart to 10 nm: the state a network is in once it has been
equilibrated, without the 1e12 pN forces of freshly thrown, crossing filaments.
"""
import ctypes

import numpy as np
import torch

from picgo_amd import abi, autograd, mech, synth

PREC = {"fp64": abi.MDN_PREC_FP64, "mixed": abi.MDN_PREC_MIXED}
CYL = 108.0   # cylinder length and neighbor-list range, nm


def _case(kind, net, fil, cyl, prec="fp64", cyl_min=None, calls=0, vecs=0):
    return {"kind": kind, "net": net, "fil": fil, "cyl": cyl, "cyl_min": cyl if cyl_min is None else cyl_min,
            "prec": prec, "calls": calls, "vecs": vecs}


def listed():
    return [
        # the smallest network of the tests (550 beads): what a call costs when there is little to do
        dict(_case("minimize", "cube", 50, 10, "fp64", calls=160), name="minimize_550"),
        # one network of ordinary size (42,000 beads) between two chemistry steps, default precision
        dict(_case("minimize", "cube", 2000, 20, "fp64", calls=160), name="minimize_42k"),
        # the benchmark's network (420,000 beads in a sphere) in the precision it is quoted in
        dict(_case("minimize", "sphere", 20000, 20, "mixed", calls=160), name="minimize_420k"),
        # a parameter sweep's or an ensemble's uneven networks in one call
        dict(_case("batch", "replicas", 48, 30, "mixed", cyl_min=5, calls=160), name="batch_48"),
        # a caller with its own integrator: forces at its own coordinates, in device memory
        dict(_case("forces", "cube", 50, 10, "fp64"), name="forces_550"),
        dict(_case("forces", "cube", 2000, 20, "mixed"), name="forces_42k"),
        dict(_case("forces", "sphere", 20000, 20, "fp64"), name="forces_420k"),
        # the lists rebuilt and read back, as analysis and the chemistry's stencils take them
        dict(_case("lists", "sphere", 20000, 20), name="lists_420k"),
        # the binder's candidate sites, searched after every minimization; filaments of uneven length
        dict(_case("binding", "cube", 2000, 26, cyl_min=14), name="binding_42k"),
        # energy, dE/dx and dE/dtheta of a parameter fit on GPU tensors
        dict(_case("autograd", "cube", 2000, 20), name="autograd_42k"),
        # Hessian-vector products: one for a Krylov iteration, a block for a block method
        dict(_case("hvp", "cube", 2000, 20, "fp64", vecs=1), name="hvp_42k"),
        dict(_case("hvp", "cube", 2000, 20, "mixed", vecs=16), name="hvp16_42k"),
    ]


def draw(rng):
    kind = rng.choice(["minimize", "minimize", "minimize", "batch", "forces", "forces", "forces", "lists", "binding",
                       "autograd", "hvp", "hvp"])
    prec = rng.choice(["fp64", "mixed"])
    if kind == "batch":
        hi = rng.randint(6, 30)
        return _case(kind, "replicas", rng.randint(4, 48), hi, prec, cyl_min=rng.randint(5, hi), calls=rng.randint(20, 160))
    net = rng.choice(["cube", "sphere"])
    # a force evaluation without allocation holds 420,000 beads of the sphere, 170,000 of the denser cube
    top = {"minimize": 20000, "forces": 20000 if net == "sphere" else 8000, "lists": 20000}.get(kind, 4000)
    fil = int(round(50 * (top / 50) ** rng.random()))
    cyl = rng.randint(2, 20)
    lo = rng.choice([cyl, rng.randint(1, cyl)])
    return _case(kind, net, fil, cyl, prec if kind in ("minimize", "forces", "hvp") else "fp64", cyl_min=lo,
                 calls=rng.randint(20, 160) if kind == "minimize" else 0,
                 vecs=rng.choice([1, 1, rng.randint(2, 16)]) if kind == "hvp" else 0)


# ---- networks -----------------------------------------------------------------------------

def _params(case, seed):
    """The generator's parameters: the presets' densities (the cube's 320 cylinders per um^3, the
    sphere's 95, 62 in the smallest), four linkers and two motors per filament."""
    fil, n = case["fil"], case["fil"] * (case["cyl"] + case["cyl_min"]) / 2
    room = CYL * (case["cyl"] + 2) / 3 ** 0.5 + 200   # the longest filament fits on a diagonal
    if case["net"] == "sphere":
        r = max(500 + CYL * (case["cyl"] + 2) / 2, 10000.0 * (n / 400000) ** (1 / 3))
        p = synth.preset(4, radius=r, box=2 * r)
    else:
        p = synth.preset(2 if case["kind"] in ("autograd", "hvp") else 1,
                         box=max(room, 2000.0 if n <= 500 else 5000.0 * (n / 40000) ** (1 / 3)))
    # uneven filaments take their lengths from the generator's stream: the same ones for every seed
    p.seed = 1000 + (seed if case["cyl_min"] == case["cyl"] else 0)
    p.n_fil, p.n_cyl_min, p.n_cyl_max = fil, case["cyl_min"], case["cyl"]
    p.n_linkers, p.n_motors = 4 * fil, 2 * fil
    return p


def _replica(case, seed, k):
    """Network k of a batch: 20 to 400 filaments of equal length, two linkers and one motor each."""
    shape, g = np.random.default_rng([case["fil"], case["cyl"], k]), np.random.default_rng([seed, k])
    p = synth.preset(3, index=k)
    p.seed = int(g.integers(1, 2 ** 31))
    nc = int(shape.integers(case["cyl_min"], case["cyl"] + 1))
    p.n_fil, p.n_cyl_min, p.n_cyl_max = int(shape.integers(20, 401)), nc, nc
    p.box = max(1000.0 * (p.n_fil * nc / 0.1) ** (1 / 3), CYL * (nc + 2) / 3 ** 0.5 + 300)
    net = synth.Network(p)
    return net, net.coord + g.normal(0.0, 2.0, net.coord.size)


def _arr(ptr, n, dtype=None):
    a = np.ctypeslib.as_array(ptr, (n,)) if n else np.zeros(0)
    return a.copy() if dtype is None else a.astype(dtype)


def _cyl_beads(d):
    """First and second bead of every cylinder, and its filament and place on it."""
    off = _arr(d.fil_bead_offset, d.n_filaments + 1, np.int64)
    beads = _arr(d.fil_beads, int(off[-1]), np.int64)
    last = np.zeros(len(beads), bool)
    last[off[1:] - 1] = True
    at = np.nonzero(~last)[0]
    fil = np.repeat(np.arange(d.n_filaments), np.diff(off) - 1)
    return beads[at], beads[at + 1], fil, at - off[fil]


def _apart(x, pairs, b1, b2, dmin=10.0, rounds=12):
    """Cylinders of the listed pairs closer than dmin pushed apart along their closest approach."""
    X = x.reshape(-1, 3).copy()
    p, q = pairs[:, 0], pairs[:, 1]
    for _ in range(rounds):
        A, u, C, v = X[b1[p]], X[b2[p]] - X[b1[p]], X[b1[q]], X[b2[q]] - X[b1[q]]
        w = A - C
        a, b, c, d, e = ((s * t).sum(1) for s, t in ((u, u), (u, v), (v, v), (u, w), (v, w)))
        s = np.clip((b * e - c * d) / np.maximum(a * c - b * b, 1e-9), 0, 1)
        t = np.clip((b * s + e) / c, 0, 1)
        s = np.clip((b * t - d) / a, 0, 1)
        n = w + s[:, None] * u - t[:, None] * v
        dist = np.sqrt((n * n).sum(1))
        k = np.nonzero(dist < dmin)[0]
        if len(k) == 0:
            break
        push = n[k] / dist[k, None] * ((dmin - dist[k]) * 0.55)[:, None]
        for ids, sign in ((b1[p[k]], 1), (b2[p[k]], 1), (b1[q[k]], -1), (b2[q[k]], -1)):
            for ax in range(3):
                X[:, ax] += np.bincount(ids, weights=sign * push[:, ax], minlength=len(X))
    return X.reshape(-1)


def _start(case, seed):
    """A network, its coordinates, and a context that holds it with its lists built there."""
    net = synth.Network(_params(case, seed))
    x = net.coord + np.random.default_rng(seed).normal(0.0, 2.0, net.coord.size)
    ffm = mech.ForceFieldManager(0)
    ffm.upload(net.desc, x)
    ffm.reset_neighbor_lists(x)
    b1, b2, _, _ = _cyl_beads(net.desc)
    x = _apart(x, ffm.neighbor_pairs(), b1, b2)
    ffm.set_coords(x)
    ffm.reset_neighbor_lists(None)
    return net, x, ffm


def _tangents(case, seed, n):
    v = np.random.default_rng(seed + 7).standard_normal((case["vecs"], n))
    return v / np.linalg.norm(v, axis=1, keepdims=True)


def _sites(case, seed, net):
    """The binder's range and free sites: four sites per cylinder, nine in ten of them free."""
    free = np.random.default_rng(seed + 9).random(net.n_cylinders * 4) < 0.9
    return abi.binding_params(np.array([0.125, 0.375, 0.625, 0.875]), 30.0, 40.0, CYL, site_free=free)


def prepare(case, seed):
    s = {"case": case, "cg": abi.default_cg_params(precision=PREC[case["prec"]], energy_call_limit=case["calls"])}
    if case["kind"] == "batch":
        made = [_replica(case, seed, k) for k in range(case["fil"])]
        s["nets"], s["x"], s["ffm"] = [m[0] for m in made], [m[1] for m in made], []
        for net, x in made:
            ffm = mech.ForceFieldManager(0)
            ffm.upload(net.desc, x)
            ffm.reset_neighbor_lists(x)
            s["ffm"].append(ffm)
        return s
    net, x, ffm = _start(case, seed)
    s.update(net=net, x=x, ffm=ffm)
    if case["kind"] in ("lists", "binding"):   # room that a caller keeps for the entries
        s["room"] = (8 if case["kind"] == "lists" else 16) * net.n_cylinders + 1000
        s["out"] = np.zeros((s["room"], 2), np.int32 if case["kind"] == "lists" else np.uint32)
        s["beads"] = np.zeros(2 * net.n_cylinders * net.desc.n_boundary, np.int32)
        s["counts"] = np.zeros(net.desc.n_boundary, np.int32)
    if case["kind"] == "forces":
        s["x_dev"] = torch.from_numpy(x).cuda()
        s["f_dev"] = torch.empty_like(s["x_dev"])
    elif case["kind"] == "binding":
        s["sites"] = _sites(case, seed, net)
    elif case["kind"] == "hvp":
        s["v"] = _tangents(case, seed, x.size)
    elif case["kind"] == "autograd":
        s["x_dev"] = torch.from_numpy(x).cuda().requires_grad_(True)
        s["theta"] = autograd.theta0(net.desc).cuda().requires_grad_(True)
    return s


# ---- the calls ----------------------------------------------------------------------------

def _result(r):
    """A minimization's energies, residuals and counts."""
    e = [r.energies_before.total, *r.energies_before.ff], [r.energies_after.total, *r.energies_after.ff]
    return {"before": np.array(e[0]), "after": np.array(e[1]), "max_force": r.grad_inf_norm,
            "counts": np.array([r.num_iter, r.num_energy_call, r.num_force_call, r.num_safe_mode, r.num_recovery])}


def _minimize(s):
    s["ffm"].reset_neighbor_lists(s["x"])
    x, f, r = s["ffm"].minimize(s["cg"], s["x"])
    return dict(_result(r), x=x, f=f)


def _batch(s):
    xs, _, res = mech.minimize_batched(s["ffm"], s["cg"], s["x"], want_forces=False)
    rs = [_result(r) for r in res]
    return {"x": xs, **{k: np.array([r[k] for r in rs]) for k in rs[0]}}


def _call(s, name, *args):
    """An entry point of the C ABI on the state's context."""
    L, h = mech.lib(), s["ffm"]._h
    st = getattr(L, name)(h, *args)
    if st:
        raise mech.MdnError(st, L.mdn_last_error(h).decode())


def _ptr(a, kind):
    return a.ctypes.data_as(ctypes.POINTER(kind))


def _forces(s):
    _call(s, "mdn_forces_noalloc", PREC[s["case"]["prec"]], ctypes.c_void_p(s["x_dev"].data_ptr()),
          ctypes.c_void_p(s["f_dev"].data_ptr()), s["x_dev"].numel())
    return s["f_dev"]


def _lists(s):
    n, m = ctypes.c_int64(), ctypes.c_int64()
    s["ffm"].reset_neighbor_lists(s["x"])
    _call(s, "mdn_nl_pairs", _ptr(s["out"], ctypes.c_int32), s["room"], ctypes.byref(n))
    _call(s, "mdn_boundary_list", _ptr(s["beads"], ctypes.c_int32), s["beads"].size, _ptr(s["counts"], ctypes.c_int32),
          ctypes.byref(m))
    return {"pairs": s["out"], "n": n.value, "beads": s["beads"], "m": m.value, "counts": s["counts"]}


def _binding(s):
    n = ctypes.c_int64()
    _call(s, "mdn_binding_pairs", ctypes.byref(s["sites"]), _ptr(s["x"], ctypes.c_double), _ptr(s["out"], ctypes.c_uint32),
          s["room"], ctypes.byref(n))
    return {"sites": s["out"], "n": n.value}


def _hvp(s):
    prec = PREC[s["case"]["prec"]]
    if s["case"]["vecs"] == 1:
        return s["ffm"].hvp(s["v"][0], s["x"], precision=prec)
    return s["ffm"].hvp_batch(s["v"], s["x"], precision=prec)


def _autograd(s):
    e = autograd.energy(s["ffm"], s["x_dev"], s["theta"])
    gx, gt = torch.autograd.grad(e, (s["x_dev"], s["theta"]))
    return {"e": e.detach(), "gx": gx, "gt": gt}


RUNS = {"minimize": _minimize, "batch": _batch, "forces": _forces, "lists": _lists, "binding": _binding, "hvp": _hvp,
        "autograd": _autograd}


def run(state):
    return RUNS[state["case"]["kind"]](state)


def work(case):
    """Bytes in and out once (coordinates, interaction tables, results) and the evaluations' FP64 operations."""
    kind = case["kind"]
    per_net = 210 if kind == "batch" else case["fil"]
    nets = case["fil"] if kind == "batch" else 1
    cyl = per_net * (case["cyl"] + case["cyl_min"]) / 2
    beads, links = cyl + per_net, (3 if kind == "batch" else 6) * per_net
    pairs = 0 if kind == "batch" else 1.3 * cyl if case["net"] == "cube" else 0.28 * cyl   # about
    tables = 24 * cyl + 28 * (cyl - per_net) + 48 * links + 40 * pairs
    energy = 20 * cyl + 40 * (cyl - per_net) + 60 * links + 450 * pairs
    x = 24 * beads
    evals = {"minimize": 1.5 * case["calls"], "batch": 1.5 * case["calls"], "forces": 2, "autograd": 4,
             "hvp": 1 + 4 * case["vecs"]}.get(kind, 0)
    out = {"minimize": 2 * x, "batch": x, "forces": x, "lists": 8 * pairs, "binding": 4 * pairs,
           "autograd": x + 24 * cyl, "hvp": 2 * case["vecs"] * x}[kind]
    flops = evals * energy + {"lists": 60 * cyl, "binding": 400 * cyl}.get(kind, 0)
    return {"bytes": nets * (x + out + (16 * cyl if kind in ("lists", "binding") else tables)), "flops": nets * flops}


# ---- 64-bit values ------------------------------------------------------------------------

class _Reference:
    """The six force fields of a network in plain torch (FP64), on the GPU."""

    def __init__(self, d, x, dev="cuda"):
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)   # noqa: E731
        b1, b2, fil, place = _cyl_beads(d)
        nc = len(b1)
        self.b1, self.b2, self.n = t(b1), t(b2), d.n_beads
        self.kexv = t(_arr(d.cyl_kexvol, nc))
        self.theta = t(np.stack([_arr(p, nc) for p in (d.cyl_kstr, d.cyl_eql, d.cyl_kbend)]))
        self.second = t(np.nonzero(place > 0)[0])   # the second cylinder of every bending term
        xl = [(ptr[i].cyl1, ptr[i].cyl2, ptr[i].pos1, ptr[i].pos2, ptr[i].kstr, ptr[i].eql)
              for ptr, n in ((d.linkers, d.n_linkers), (d.motors, d.n_motors)) for i in range(n)]
        xl = np.array(xl).reshape(-1, 6)
        self.n_link = d.n_linkers
        self.xc = t(xl[:, :2].astype(np.int64))
        self.xp = t(xl[:, 2:])
        x = t(x).reshape(-1, 3)
        mid = 0.5 * (x[self.b1] + x[self.b2])
        # the half list of cylinders c > c' with midpoints in range, same-filament neighbours left out
        rsq, fil, place, found = float(np.float32(d.exvol_rmax) ** 2), t(fil), t(place), []
        rows = max(1, 50_000_000 // max(1, nc))
        for a in range(0, nc, rows):
            m = mid[a:a + rows, None, :]
            d2 = ((mid[None, :min(nc, a + rows)] - m) ** 2).sum(2)
            i, j = torch.nonzero(d2 <= rsq, as_tuple=True)
            i = i + a
            ok = (i > j) & ((fil[i] != fil[j]) | ((place[i] - place[j]).abs() > 2))
            found.append(torch.stack([i[ok], j[ok]]))
            del d2
        self.pairs = torch.cat(found, 1)
        # boundary interactions: every cylinder in range adds its second bead, a minus end its first too
        self.bnd = []
        for e in range(d.n_boundary):
            el = d.boundary[e]
            inside = self._distance(el, mid) < d.boundary_cutoff
            self.bnd.append((el, torch.cat([self.b2[inside], self.b1[inside & (place == 0)]])))

    @staticmethod
    def _distance(el, x):
        p = list(el.p)
        if el.kind == abi.MDN_BND_PLANE:
            n = x.new_tensor(p[:3])
            return (x @ n + p[3]) / n.norm()
        return p[3] - (x - x.new_tensor(p[:3])).norm(dim=1)

    @staticmethod
    def _pair_energy(c1, c2, c3, c4, ks):
        """Repulsion of two segments, ks / |r - r'|^4 integrated over both, in closed form."""
        dot = lambda a, b: (a * b).sum(1)   # noqa: E731
        u, v, w = c2 - c1, c4 - c3, c1 - c3
        a, b, c, d, e, f = dot(u, u), dot(v, v), dot(w, w), dot(u, v), dot(u, w), dot(v, w)
        w14, w32 = c4 - c1, c2 - c3
        g, h, i = dot(u, w14), dot(v, w32), dot(v, w14)
        root = lambda p, q: torch.sqrt((torch.sqrt(p) + q) * (torch.sqrt(p) - q))   # noqa: E731
        A, B = root(a * c, e), root(b * c, f)
        E, F = root(a * dot(w14, w14), g), root(b * dot(w32, w32), h)
        C, D, G = d * e - a * f, b * e - d * f, d * g - a * i
        J = -dot(torch.linalg.cross(u, v), w) ** 2
        at = torch.atan
        s = (C / A * (at((a + e) / A) - at(e / A)) + G / E * (at((a + e - d) / E) - at((e - d) / E))
             + D / B * (at(f / B) - at((f - b) / B)) + (C + G - D) / F * (at((d + f) / F) - at((d + f - b) / F)))
        return 0.5 * ks / J * s

    def _pair_beads(self, x):
        i, j = self.pairs
        return x[self.b1[i]], x[self.b2[i]], x[self.b1[j]], x[self.b2[j]]

    def _pair_k(self, theta):
        i, j = self.pairs
        return self.kexv[i] * theta[1][i] * theta[1][j]

    def _bonded(self, x, theta):
        r = x[self.b2] - x[self.b1]
        L = r.norm(dim=1)
        stretch = 0.5 * theta[0] * (L - theta[1]) ** 2
        u = r / L[:, None]
        bend = theta[2][self.second] * (1 - (u[self.second - 1] * u[self.second]).sum(1))
        p1, p2, k, L0 = self.xp.T
        at = lambda c, p: x[self.b1[c]] * (1 - p)[:, None] + x[self.b2[c]] * p[:, None]   # noqa: E731
        link = 0.5 * k * ((at(self.xc[:, 1], p2) - at(self.xc[:, 0], p1)).norm(dim=1) - L0) ** 2
        wall = sum(el.krep * torch.exp(-self._distance(el, x[b]) / el.slen).sum() for el, b in self.bnd)
        return stretch.sum(), bend.sum(), link[:self.n_link].sum(), link[self.n_link:].sum(), wall

    def energies(self, x, theta):
        s, b, link, motor, wall = self._bonded(x, theta)
        pair = self._pair_energy(*self._pair_beads(x), self._pair_k(theta)).sum()
        return [s, b, link, motor, pair, wall]

    def forces(self, x):
        """-dE/dx; the excluded-volume forces of nearly coplanar pairs at a geometry whose second
        bead is moved 0.01 nm along the plane's normal, as the model defines them."""
        theta = self.theta
        f = -torch.func.grad(lambda y: sum(self._bonded(y, theta)))(x)
        if self.pairs.shape[1] == 0:
            return f
        c1, c2, c3, c4 = self._pair_beads(x)
        n = torch.linalg.cross(c2 - c1, c3 - c1)
        n = n / n.norm(dim=1, keepdim=True)
        flat = ((c4 - c1) / (c4 - c1).norm(dim=1, keepdim=True) * n).sum(1).abs() < 0.1
        c2 = torch.where(flat[:, None], c2 + 0.01 * n, c2)
        ks = self._pair_k(theta)
        g = torch.func.grad(lambda *c: self._pair_energy(*c, ks).sum(), argnums=(0, 1, 2, 3))(c1, c2, c3, c4)
        i, j = self.pairs
        for b, gb in zip((self.b1[i], self.b2[i], self.b1[j], self.b2[j]), g):
            f = f.index_add(0, b, -gb)
        return f


def exact(case, seed):
    """64-bit values. A minimization's path follows every rounding of its many evaluations (two
    starts 1e-12 nm apart end 1e-3 nm apart), so only its energies at the start have one."""
    kind = case["kind"]
    if kind in ("lists", "binding"):
        return None
    if kind == "batch":
        made = [_replica(case, seed, k) for k in range(case["fil"])]
        before = [_Reference(net.desc, x).energies for net, x in made]
        before = [f(torch.as_tensor(x, device="cuda").reshape(-1, 3), f.__self__.theta) for f, (_, x) in zip(before, made)]
        return {"x": [None] * case["fil"], "before": np.array([[float(sum(e)), *map(float, e)] for e in before]),
                "after": None, "max_force": None, "counts": None}
    net, x, ffm = _start(case, seed)
    ffm.close()
    ref = _Reference(net.desc, x)
    xt = torch.as_tensor(x, device="cuda").reshape(-1, 3)
    if kind == "minimize":
        e = [float(v) for v in ref.energies(xt, ref.theta)]
        return {"before": np.array([sum(e), *e]), "after": None, "max_force": None, "counts": None, "x": None, "f": None}
    if kind == "forces":
        return ref.forces(xt).reshape(-1)
    if kind == "autograd":
        theta = ref.theta.clone().requires_grad_(True)
        e = sum(ref.energies(xt, theta))
        return {"e": e.detach(), "gx": -ref.forces(xt).reshape(-1), "gt": torch.autograd.grad(e, theta)[0]}
    v = torch.as_tensor(_tangents(case, seed, x.size), device="cuda")
    h = torch.stack([-torch.func.jvp(ref.forces, (xt,), (w.reshape(-1, 3),))[1].reshape(-1) for w in v])
    return h[0] if case["vecs"] == 1 else h
