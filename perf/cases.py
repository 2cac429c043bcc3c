"""The work that a user of this library has it do, as cases that can be timed.

Particles are drawn on the GPU from the distributions of nbodylib_amd.datagen: a uniform box, or half a uniform
background and half NFW halos (2000 in sets of a million or more), with bulk and internal velocities.  Trees are what
a program keeps from call to call, so they are made in prepare() except where the case is the whole snapshot.

A case holds its kind (one of KINDS), the particle count n, the neighbour count k and the kind's options.
"""
import math

import numpy as np
import torch

import nbodylib_amd as nb
from nbodylib_amd.device import DeviceTree, SPHDensity

BOX = 100.0      # side of the clustered box
FORMS = {"plain": nb.FORM_PLAIN, "mixed": nb.FORM_MIXED}
PAIRS = 1.1e11   # all-pairs distances that exact() computes at most


def listed():
    return [
        # one time step of a small run: every particle's neighbours in a periodic box, latency above all
        {"name": "knn_periodic_4k", "kind": "knn", "n": 4096, "k": 32, "form": "plain", "set": "uniform", "periodic": True},
        # neighbour table with distances of a mid-sized snapshot, odd sizes, FP32 search
        {"name": "knn_rows_1m", "kind": "knn", "n": 1000003, "k": 20, "form": "mixed", "set": "clustered", "periodic": False},
        # CalcDensity of the drop-in's default form (FP64 throughout)
        {"name": "density_plain_2m", "kind": "density", "n": 2097152, "k": 32, "form": "plain", "variant": "symmetric"},
        # the headline: neighbours, density and smoothing length of a large snapshot in one call
        {"name": "knn_density_16m", "kind": "knn_density", "n": 16777216, "k": 32, "form": "mixed"},
        # phase-space density of a halo finder's input
        {"name": "phase_density_2m", "kind": "phase", "n": 2097152, "k": 64, "form": "mixed"},
        # group catalogue of a large snapshot whose tree is kept
        {"name": "fof_16m", "kind": "fof", "n": 16777216},
        # phase-space groups (the substructure search)
        {"name": "fof6d_1m5", "kind": "fof6d", "n": 1500007},
        # a snapshot from raw particles to its groups: tree build and FOF, nothing kept
        {"name": "snapshot_fof_2m", "kind": "snapshot", "n": 2000003},
        # one optimisation step through the density: forward and backward over a stored list, input order
        {"name": "adjoint_1m", "kind": "adjoint", "n": 1048576, "k": 32},
        # the same where the list does not fit: recomputed per block of tree slots
        {"name": "adjoint_tree_1m", "kind": "adjoint_tree", "n": 1048576, "k": 32, "form": "mixed", "block": 262144},
        # densities at probe positions, host arrays in and out
        {"name": "points_100k", "kind": "points", "n": 1000000, "m": 100003, "k": 32},
        # velocity dispersion field, host arrays out
        {"name": "smooth_disp_500k", "kind": "smooth", "n": 524288, "k": 32},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(KINDS)
    k = rng.choice([8, 16, 20, 24, 32, 33, 40, 48, 64])
    form = rng.choice(["plain", "mixed"])
    if kind == "knn":
        periodic = rng.random() < 0.5
        return {"kind": kind, "n": _size(rng, 4096, 2000000), "k": k, "form": form,
                "set": rng.choice(["uniform", "clustered"]), "periodic": periodic}
    if kind == "density":
        return {"kind": kind, "n": _size(rng, 4096, 4000000), "k": k, "form": form,
                "variant": rng.choice(["symmetric", "gather"])}
    if kind == "knn_density":
        return {"kind": kind, "n": _size(rng, 4096, 16777216), "k": rng.choice([16, 20, 24, 32]), "form": "mixed"}
    if kind == "phase":
        return {"kind": kind, "n": _size(rng, 4096, 2000000), "k": k, "form": "mixed"}
    if kind == "fof":
        return {"kind": kind, "n": _size(rng, 4096, 16777216)}
    if kind == "fof6d":
        return {"kind": kind, "n": _size(rng, 4096, 2000000)}
    if kind == "snapshot":
        return {"kind": kind, "n": _size(rng, 4096, 4000000)}
    if kind == "adjoint":
        return {"kind": kind, "n": _size(rng, 4096, 2000000), "k": k}
    if kind == "adjoint_tree":
        n = _size(rng, 4096, 2000000)
        return {"kind": kind, "n": n, "k": k, "form": form, "block": _size(rng, max(2048, n // 8), n)}
    if kind == "points":
        return {"kind": kind, "n": _size(rng, 4096, 2000000), "m": _size(rng, 64, 200000), "k": k}
    return {"kind": "smooth", "n": _size(rng, 4096, 600000), "k": k}


# ------------------------------------------------------------------ particles
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 12345)
    return g


def _uniform(n, g, side):
    return torch.rand((3, n), generator=g, device="cuda", dtype=torch.float64) * side


def _clustered(n, g, with_vel=False):
    """(3, n) positions [and velocities]: datagen.clustered's recipe on the GPU, with fewer halos in small sets, so
    that the halos of a small set still hold groups."""
    nhalo = max(4, min(2000, n // 512))
    def rand(m):
        return torch.rand(m, generator=g, device="cuda", dtype=torch.float64)

    def normal(shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)

    nbg = n // 2
    nh = n - nbg
    centres = rand(3 * nhalo).view(3, nhalo) * BOX
    conc = 5.0 + 10.0 * rand(nhalo)
    rs = 0.05 + 0.45 * rand(nhalo)
    a1 = -0.9
    mass = (1.0 + rand(nhalo) * (1e3 ** a1 - 1.0)) ** (1.0 / a1)
    share = torch.cumsum(mass, 0) / mass.sum() * nh
    edge = torch.round(share).to(torch.int64)
    edge[-1] = nh
    hid = torch.searchsorted(edge, torch.arange(nh, device="cuda"), right=True)
    c = conc[hid]
    mu = lambda x: torch.log1p(x) - x / (1.0 + x)  # noqa: E731  (enclosed NFW mass)
    target = rand(nh) * mu(c)
    lo, hi = torch.zeros_like(c), c.clone()
    for _ in range(45):
        mid = 0.5 * (lo + hi)
        below = mu(mid) < target
        lo, hi = torch.where(below, mid, lo), torch.where(below, hi, mid)
    r = 0.5 * (lo + hi) * rs[hid]
    v = normal((3, nh))
    v /= v.norm(dim=0)
    pos = torch.empty((3, n), device="cuda", dtype=torch.float64)
    pos[:, :nbg] = _uniform(nbg, g, BOX)
    pos[:, nbg:] = centres[:, hid] + r * v
    pos = torch.remainder(pos, BOX)
    pos[pos >= BOX] = 0.0
    if not with_vel:
        return pos
    vel = torch.empty((3, n), device="cuda", dtype=torch.float64)
    vel[:, :nbg] = 300.0 * normal((3, nbg))
    sig = 300.0 * (mass / mass.max()) ** (1.0 / 3.0)
    vel[:, nbg:] = 300.0 * normal((3, nhalo))[:, hid] + normal((3, nh)) * sig[hid]
    return pos, vel


def _masses(n, g):
    return torch.exp(0.3 * torch.randn(n, generator=g, device="cuda", dtype=torch.float64) - 0.045) / n


def _link(n):
    return 0.2 * BOX / n ** (1.0 / 3.0)


def _inputs(case, seed):
    """What the case's particles are, on the GPU."""
    g, n, kind = _gen(seed), case["n"], case["kind"]
    if kind == "knn" and case["set"] == "uniform":
        return {"pos": _uniform(n, g, 1.0), "side": 1.0}
    if kind in ("phase", "fof6d"):
        pos, vel = _clustered(n, g, with_vel=True)
        sx = pos.std(dim=1, keepdim=True)
        return {"pos": pos / sx, "vel": vel / vel.std(dim=1, keepdim=True), "sx": float(sx.mean())}
    if kind == "smooth":
        pos, vel = _clustered(n, g, with_vel=True)
        return {"pos": pos, "vel": vel}
    d = {"pos": _clustered(n, g), "side": BOX}
    if kind in ("adjoint", "adjoint_tree"):
        d["mass"] = _masses(n, g)
        d["g"] = torch.randn(n, generator=g, device="cuda", dtype=torch.float64)
    if kind == "points":
        # half anywhere in the box, half near particles, in no order
        m = case["m"]
        x = _uniform(m, g, BOX)
        at = torch.randint(n, (m - m // 2,), generator=g, device="cuda")
        x[:, m // 2:] = d["pos"][:, at] + 0.02 * torch.randn((3, at.numel()), generator=g, device="cuda", dtype=torch.float64)
        d["x"] = x[:, torch.randperm(m, generator=g, device="cuda")].contiguous()
    return d


def _host(t):
    return np.ascontiguousarray(t.t().cpu().numpy())


# ------------------------------------------------------------------ the calls
def prepare(case, seed):
    d, n, kind = _inputs(case, seed), case["n"], case["kind"]
    out = lambda *shape, dtype=torch.float64: torch.empty(shape, device="cuda", dtype=dtype)  # noqa: E731
    s = {"case": case}
    if kind == "knn":
        s["tree"] = DeviceTree(d["pos"], kerntype=nb.KSPH, period=d["side"] if case["periodic"] else None,
                               form=FORMS[case["form"]])
        s["nn"], s["d2"] = out(n, case["k"], dtype=torch.int32), out(n, case["k"])
    elif kind in ("density", "knn_density"):
        s["tree"] = DeviceTree(d["pos"], kerntype=nb.KSPH, period=BOX, form=FORMS[case["form"]])
        s["rho"], s["h"] = out(n), out(n)
        if kind == "knn_density":
            s["nn"] = out(n, case["k"], dtype=torch.int32)
    elif kind == "phase":
        s["tree"] = DeviceTree(d["pos"], vel=d["vel"], treetype=nb.TPHS, kerntype=nb.KSPH, aniso=-1,
                               form=FORMS[case["form"]])
        s["rho"], s["h"] = out(n), out(n)
    elif kind == "fof":
        s["tree"] = DeviceTree(d["pos"], kerntype=nb.KSPH, period=BOX)
        s["labels"] = out(n, dtype=torch.int32)
    elif kind == "fof6d":
        s["tree"] = DeviceTree(d["pos"], vel=d["vel"], treetype=nb.TPHS, kerntype=nb.KSPH, aniso=-1)
        s6 = (_link(n) / d["sx"]) ** 2
        s["params"] = [nb.TPHS, s6, 0.01, 0, 0, 0, s6, 0.01]
        s["labels"] = out(n, dtype=torch.int32)
    elif kind == "snapshot":
        s["pos"], s["labels"] = d["pos"], out(n, dtype=torch.int32)
    elif kind == "adjoint":
        tree = DeviceTree(d["pos"], mass=d["mass"], kerntype=nb.KSPH, form=nb.FORM_MIXED)
        nbr, d2 = out(n, case["k"], dtype=torch.int32), out(n, case["k"])
        tree.knn(case["k"], nbr, d2, layout=nb.LAYOUT_BY_ID)
        s["nbr"], s["g"] = nbr, d["g"]
        s["pos"], s["mass"] = d["pos"].requires_grad_(), d["mass"].requires_grad_()
    elif kind == "adjoint_tree":
        s["tree"] = DeviceTree(d["pos"], mass=d["mass"], kerntype=nb.KSPH, form=FORMS[case["form"]])
        s["g"], s["rho"], s["h"], s["dpos"], s["dmass"] = d["g"], out(n), out(n), out(3, n), out(n)
    elif kind == "points":
        s["tree"] = nb.KDTree(_host(d["pos"]), kerntype=nb.KSPH)
        s["x"] = _host(d["x"])
    else:
        s["tree"] = nb.KDTree(_host(d["pos"]), vel=_host(d["vel"]), kerntype=nb.KSPH)
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "knn":
        s["tree"].knn(c["k"], s["nn"], s["d2"], variant=nb.KNN_FINDNEAREST, layout=nb.LAYOUT_BY_ID)
        return s["nn"], s["d2"]
    if kind == "density":
        s["tree"].density(c["k"], s["rho"], s["h"], variant=nb.DENS_GATHER if c["variant"] == "gather" else nb.DENS_SYMMETRIC)
        return s["rho"], s["h"]
    if kind == "knn_density":
        s["tree"].knn_density(c["k"], s["nn"], s["rho"], s["h"])
        return s["nn"], s["rho"], s["h"]
    if kind == "phase":
        s["tree"].density(c["k"], s["rho"], s["h"])
        return s["rho"], s["h"]
    if kind == "fof":
        return s["labels"], s["tree"].fof(_link(c["n"]), 8, s["labels"])
    if kind == "fof6d":
        return s["labels"], s["tree"].fof_criterion(nb.FOF_CMP_6D, s["params"], 8, s["labels"])
    if kind == "snapshot":
        tree = DeviceTree(s["pos"], kerntype=nb.KSPH, period=BOX)
        return s["labels"], tree.fof(_link(c["n"]), 8, s["labels"])
    if kind == "adjoint":
        rho = SPHDensity.apply(s["pos"], s["mass"], s["nbr"])
        dpos, dmass = torch.autograd.grad(rho, (s["pos"], s["mass"]), s["g"])
        return rho, dpos, dmass
    if kind == "adjoint_tree":
        s["tree"].sph_density(c["k"], s["rho"], s["h"], block_rows=c["block"])
        s["tree"].sph_density_adjoint(c["k"], s["g"], s["dpos"], s["dmass"], block_rows=c["block"])
        return s["rho"], s["h"], s["dpos"], s["dmass"]
    if kind == "points":
        return s["tree"].CalcDensityPosition(s["x"], c["k"], return_h=True)
    return s["tree"].CalcSmoothVelDisp(c["k"])


def work(case):
    """Each input once, each output once (positions and masses in FP64, neighbours and labels in 32 bits); the
    arithmetic is one distance and one weight per neighbour."""
    n, k, kind = case["n"], case.get("k", 0), case["kind"]
    pair = 20.0  # distance, kernel and sum of one neighbour
    if kind == "knn":
        return {"bytes": n * (24 + 12 * k), "flops": 8.0 * n * k}
    if kind == "density":
        return {"bytes": n * (32 + 16), "flops": pair * n * k}
    if kind == "knn_density":
        return {"bytes": n * (32 + 16 + 4 * k), "flops": pair * n * k}
    if kind == "phase":
        return {"bytes": n * (56 + 16), "flops": 1.5 * pair * n * k}
    if kind == "fof":
        return {"bytes": n * 28, "flops": 8.0 * n}
    if kind == "fof6d":
        return {"bytes": n * 52, "flops": 17.0 * n}
    if kind == "snapshot":
        return {"bytes": n * 28, "flops": 8.0 * n}
    if kind == "adjoint":  # forward reads pos, mass and the list; backward the same and g
        return {"bytes": n * (32 + 4 * k + 8 + 40 + 4 * k + 32), "flops": 3 * pair * n * k}
    if kind == "adjoint_tree":
        return {"bytes": n * (32 + 16 + 40 + 32), "flops": 3 * pair * n * k}
    if kind == "points":
        return {"bytes": case["m"] * (24 + 16) + 32 * n, "flops": pair * case["m"] * k}
    return {"bytes": n * (56 + 96), "flops": 3 * pair * n * k}


# ------------------------------------------------------------------ the same in 64 bits, by all pairs
def _dist2(q, x):
    s = None
    for d in range(q.shape[0]):
        t = q[d][:, None] - x[d][None, :]
        s = t * t if s is None else s + t * t
    return s


def _nearest(q, x, k, drop_self):
    """(d2, index) of the k nearest of x to each q; drop_self: q is x, and d2 == 0 is no neighbour."""
    m, n = q.shape[1], x.shape[1]
    step = max(1, int(2.5e8 // n))
    d2, at = torch.empty((m, k), device="cuda", dtype=torch.float64), torch.empty((m, k), device="cuda", dtype=torch.int64)
    for a in range(0, m, step):
        d = _dist2(q[:, a:a + step], x)
        if drop_self:
            d[d == 0.0] = 1e32
        d2[a:a + step], at[a:a + step] = torch.topk(d, k, dim=1, largest=False)
    return d2, at


def _nearest_images(x, side, k):
    """FindNearest of the reference in a periodic box: k + 1 kept over the box and its images in turn (an image is
    taken where its offset, squared or not as the reference has it, lies within the kept radius), the first dropped."""
    n = x.shape[1]
    kept = torch.full((n, k + 1), 1e32, device="cuda", dtype=torch.float64)
    low = x < side / 2.0
    far = torch.where(low, x + side, x - side)
    wall = torch.where(low, x, -far)
    step = max(1, int(1.5e8 // n))
    for dims in ((), (0,), (1,), (2,), (0, 1), (0, 2), (1, 2), (0, 1, 2)):
        q = x.clone()
        for d in dims:
            q[d] = far[d]
        kth = kept[:, -1]
        if not dims:
            take = torch.ones(n, device="cuda", dtype=torch.bool)
        elif len(dims) == 1:
            take = torch.sqrt(kth) > wall[dims[0]]
        else:
            take = kth > torch.sqrt(sum(wall[d] ** 2 for d in dims))
        rows = take.nonzero()[:, 0]
        for a in range(0, rows.numel(), step):
            r = rows[a:a + step]
            d = torch.cat([kept[r], _dist2(q[:, r], x)], 1)
            kept[r] = torch.topk(d, k + 1, dim=1, largest=False)[0]
    return kept[:, 1:]


def _kernel(r, h, nd):
    """The table of the cubic spline (1000 entries) and its linear interpolation."""
    res = 1000
    norm = 1.0 / nd * math.pi ** (-nd / 2.0) * math.gamma(nd / 2.0 + 1.0)
    norm *= nd * (nd + 1.0) * (nd + 2.0) * (nd + 3.0) / (6.0 * (2.0 ** (nd + 1) - 1.0))
    step = 2.0 / (res - 1)
    q = torch.arange(res, device="cuda", dtype=torch.float64) * step
    tab = norm * torch.where(q <= 1.0, 1.0 - 0.75 * (2.0 - q) * q * q,
                             torch.where(q <= 2.0, 0.25 * (2.0 - q) ** 3, torch.zeros_like(q)))
    u = r / h
    f = u * 0.5 * (res - 1)
    i = torch.clamp(f.to(torch.int64), 0, res - 2)
    w = tab[i] + (tab[i + 1] - tab[i]) * (u - step * i.to(torch.float64)) / step
    return torch.where(f < res - 1, w, tab[res - 1])


def _spline(q):
    t, s = torch.clamp(2.0 - q, min=0.0), torch.clamp(1.0 - q, min=0.0)
    return 0.25 * t ** 3 - s ** 3


def _symmetric(x, mass, nbr):
    """Density over a list whose last column sets h, by the analytic spline."""
    d = torch.sqrt(sum((x[c][:, None] - x[c][nbr]) ** 2 for c in range(3)))
    h = 0.5 * d[:, -1]
    w = 0.5 / math.pi * _spline(d / h[:, None]) / h[:, None] ** 3
    return (w * mass[nbr]).sum(1).index_add(0, nbr.reshape(-1), (w * mass[:, None]).reshape(-1)), h


def _grads(x, mass, nbr, g):
    x, mass = x.detach().requires_grad_(), mass.detach().requires_grad_()
    rho, h = _symmetric(x, mass, nbr)
    return (rho.detach(), h.detach()) + torch.autograd.grad(rho, (x, mass), g)


def exact(case, seed):
    n, k, kind = case["n"], case.get("k", 0), case["kind"]
    if kind in ("fof", "fof6d", "snapshot"):
        return None  # labels alone: nothing is rounded
    if kind == "adjoint":
        s = prepare(case, seed)
        rho, _, dx, dm = _grads(s["pos"], s["mass"], s["nbr"].long(), s["g"])
        return rho, dx, dm
    if (case["m"] if kind == "points" else n) * float(n) > (PAIRS / 4 if case.get("periodic") else PAIRS):
        return None
    d = _inputs(case, seed)
    x = d["pos"]
    if kind == "knn":
        return None, _nearest_images(x, d["side"], k) if case["periodic"] else _nearest(x, x, k, True)[0]
    if kind == "points":
        d2, _ = _nearest(d["x"], x, k, False)
        h = 0.5 * torch.sqrt(d2[:, -1])
        rho = (_kernel(torch.sqrt(d2), h[:, None], 3) / n).sum(1) / h ** 3
        return rho.cpu().numpy(), h.cpu().numpy()
    if kind == "smooth":
        return _dispersion(x, d["vel"], k)
    if kind == "adjoint_tree":
        _, at = _nearest(x, x, k, True)
        rho, h, dx, dm = _grads(x, d["mass"], at, d["g"])
        return rho, h, dx, dm
    q = torch.cat([x, d["vel"]]) if kind == "phase" else x
    rho, h, _, _ = _density(q, k, gather=case.get("variant") == "gather")
    return (None, rho, h) if kind == "knn_density" else (rho, h)


def _density(x, k, gather=False):
    nd, n = x.shape
    d2, at = _nearest(x, x, k, True)
    h = 0.5 * torch.sqrt(d2[:, -1])
    w = _kernel(torch.sqrt(d2), h[:, None], nd) / h[:, None] ** nd / n
    if gather:
        return w.sum(1), h, at, w
    w = 0.5 * w
    return w.sum(1).index_add(0, at.reshape(-1), w.reshape(-1)), h, at, w


def _dispersion(x, v, k):
    n = x.shape[1]
    rho, _, at, w = _density(x, k)  # w holds the pair's half weight times the (equal) mass
    mine, theirs = w / rho[at], w / rho[:, None]
    flat = at.reshape(-1)
    mean = torch.stack([(mine * v[c][at]).sum(1).index_add(0, flat, (theirs * v[c][:, None]).reshape(-1)) for c in range(3)])
    disp = torch.empty((n, 3, 3), device="cuda", dtype=torch.float64)
    for a in range(3):
        for b in range(a, 3):
            s = (mine * (v[a][at] - mean[a][:, None]) * (v[b][at] - mean[b][:, None])).sum(1)
            t = theirs * (v[a][:, None] - mean[a][at]) * (v[b][:, None] - mean[b][at])
            disp[:, a, b] = disp[:, b, a] = s.index_add(0, flat, t.reshape(-1))
    return mean.t().contiguous().cpu().numpy(), disp.cpu().numpy()


KINDS = ["knn", "density", "knn_density", "phase", "fof", "fof6d", "snapshot", "adjoint", "adjoint_tree", "points", "smooth"]
