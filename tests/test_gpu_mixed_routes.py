"""The precision form's own kernel, in the calls that run it: rows without
distances and the fused search and density at any size, rows with distances
and the spline density above the sizes up to which a wave searches for one
query.  Each test asserts from the launch counts that the kernel ran."""
import contextlib

import numpy as np
import pytest

import oracle
from nbodylib_amd import datagen

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def _runs_mixed():
    import torch

    import nbodylib_amd as nb

    nb.prof_reset()
    nb.prof_enable(True)
    try:
        yield
        torch.cuda.synchronize()
    finally:
        nb.prof_enable(False)
    assert nb.prof_get("k_knn_mixed")[1] > 0, "the FP32 kernel did not run"


def _dev(a):
    import torch

    return torch.tensor(np.ascontiguousarray(a.T), dtype=torch.float64, device="cuda")


def _lattice(g):
    ax = np.arange(g) + 0.5
    p = np.stack(np.meshgrid(ax, ax, ax, indexing="ij"), -1).reshape(-1, 3)
    return p[np.random.default_rng(g).permutation(len(p))]  # IDs in no spatial order


def _rows(t, k, layout, d2=True):
    import torch

    nn = torch.full((t.n, k), -7, dtype=torch.int32, device="cuda")
    dd = torch.full((t.n, k), -1.0, dtype=torch.float64, device="cuda") if d2 else None
    t.knn(k, nn, dd, variant=3, layout=layout)
    torch.cuda.synchronize()
    return nn, dd


# (k, clustered n, lattice side): n above 163840 + 8192 k, odd, in no whole waves
@pytest.mark.parametrize("k,n,g", [(1, 172101, 56), (7, 221301, 61), (32, 426001, 76)])
@pytest.mark.parametrize("kind", ["clustered", "lattice"])
def test_rows_with_distances(gpu, kind, k, n, g):
    import torch

    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree

    pos = _lattice(g) if kind == "lattice" else datagen.clustered(n, 100.0, nhalo=60, seed=k)[0]
    print(f"mixed routes rows {kind} n={len(pos)} k={k}", flush=True)
    p = _dev(pos)
    tm = DeviceTree(p, kerntype=nb.KSPH, form=nb.FORM_MIXED)
    tp = DeviceTree(p, kerntype=nb.KSPH)
    for layout in (nb.LAYOUT_BY_ID, nb.LAYOUT_BY_SLOT):
        with _runs_mixed():
            nm, dm = _rows(tm, k, layout)
        assert tm.last_fallbacks() < tm.n
        npl, dp = _rows(tp, k, layout)
        assert torch.equal(dm, dp) and torch.equal(nm, npl)


def test_phase_rows_with_distances(gpu):
    import torch

    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree

    n, k = 1048577 + 70, 5
    print(f"mixed routes phase rows n={n} k={k}", flush=True)
    x, v, _ = datagen.clustered(n, 1.0, nhalo=200, seed=9, with_vel=True)
    x, v = _dev(x / x.std()), _dev(v / v.std())
    rows = []
    for form in (nb.FORM_MIXED, nb.FORM_PLAIN):
        t = DeviceTree(x, vel=v, treetype=nb.TPHS, aniso=-1, kerntype=nb.KSPH, form=form)
        with _runs_mixed() if form == nb.FORM_MIXED else contextlib.nullcontext():
            rows.append([_rows(t, k, layout) for layout in (0, 1)])
        del t
    for (nm, dm), (npl, dp) in zip(*rows):
        assert torch.equal(dm, dp) and torch.equal(nm, npl)


# sums of a few hundred products in any order
@pytest.mark.parametrize("k,n", [(2, 143501), (8, 180301), (32, 330001)])
def test_spline_forward(gpu, k, n):
    import torch

    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree, sph_density

    print(f"mixed routes spline n={n} k={k}", flush=True)
    p = _dev(datagen.clustered(n, 1.0, nhalo=60, seed=k)[0])
    m = torch.tensor(datagen.lognormal_masses(n, k), device="cuda")
    nn, _ = _rows(DeviceTree(p, mass=m, kerntype=nb.KSPH), k, nb.LAYOUT_BY_ID)
    ro, ho = sph_density(p, m, nn)
    t = DeviceTree(p, mass=m, kerntype=nb.KSPH, form=nb.FORM_MIXED)
    rho, h = torch.full_like(ro, -1.0), torch.full_like(ho, -1.0)
    with _runs_mixed():
        t.sph_density(k, rho, h)
    assert torch.equal(h, ho)
    assert float((rho / ro - 1.0).abs().max()) < 1e-12


def test_adjoint_blocks(gpu):
    """Two whole blocks above the line (the second at row0 > 0), then a partial
    one below it; and every slot at once."""
    import torch

    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree, SPHDensity

    k, block = 8, 245760
    n = 2 * block + 8517
    print(f"mixed routes adjoint n={n} k={k}", flush=True)
    p = _dev(datagen.clustered(n, 100.0, nhalo=150, seed=12)[0])
    m = torch.tensor(datagen.lognormal_masses(n, 12), device="cuda")
    nn, _ = _rows(DeviceTree(p, mass=m, kerntype=nb.KSPH), k, nb.LAYOUT_BY_ID)
    pg, mg = p.clone().requires_grad_(), m.clone().requires_grad_()
    rho = SPHDensity.apply(pg, mg, nn)
    g = (1.0 / rho).detach()
    rho.backward(g)
    t = DeviceTree(p, mass=m, kerntype=nb.KSPH, form=nb.FORM_MIXED)
    for rows in (block, n):
        dp, dm = torch.full_like(p, 7.0), torch.full_like(m, 7.0)
        with _runs_mixed():
            t.sph_density_adjoint(k, g, dp, dm, block_rows=rows)
        for a, b in ((dp, pg.grad), (dm, mg.grad)):
            assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())


def test_duplicates_fall_back(gpu):
    """Three particles at one point cannot be settled in FP32 nor by the
    candidates kept: those queries, and not all, are searched again in FP64."""
    import torch

    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree

    n, k = 3000, 16
    print(f"mixed routes duplicates n={n} k={k}", flush=True)
    pos = datagen.uniform(n, 1.0, 24)
    pos[1::7] = pos[0::7][: len(pos[1::7])]
    pos[2::7] = pos[0::7][: len(pos[2::7])]
    t = DeviceTree(_dev(pos), kerntype=nb.KSPH, form=nb.FORM_MIXED)
    nn = torch.empty((n, k), dtype=torch.int32, device="cuda")
    rho, h = (torch.empty(n, dtype=torch.float64, device="cuda") for _ in range(2))
    with _runs_mixed():
        t.knn_density(k, nn, rho, h)
    assert 3 * (n // 7) <= t.last_fallbacks() < n
    order = t.order().cpu().numpy()
    bi, bd = oracle.knn_brute(pos, k, mode=0)
    assert np.array_equal(np.sort(order[nn.cpu().numpy()], 1), np.sort(bi[order], 1))
    assert np.array_equal(h.cpu().numpy(), 0.5 * np.sqrt(bd[:, -1]))
    ro = oracle.Tree(pos, b=16, kerntype=oracle.KSPH).calc_density(k)
    assert np.max(np.abs(rho.cpu().numpy() / ro - 1.0)) < 1e-12


@pytest.mark.parametrize("band", [1e-12, 1e-5, 1e-3, 3e-2])
def test_recheck_band(gpu, band):
    """A wider re-check band sends more entries to FP64 and changes no set."""
    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree

    n, k = 30011, 32
    print(f"mixed routes recheck_rel={band} n={n} k={k}", flush=True)
    p = _dev(datagen.clustered(n, 100.0, nhalo=40, seed=87)[0])
    t = DeviceTree(p, kerntype=nb.KSPH, form=nb.FORM_MIXED, recheck_rel=band)
    with _runs_mixed():
        nn, _ = _rows(t, k, nb.LAYOUT_BY_ID, d2=False)
    want, _ = _rows(DeviceTree(p, kerntype=nb.KSPH), k, nb.LAYOUT_BY_ID)
    assert (nn.sort(1).values == want.sort(1).values).all()


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("kind", ["clustered", "lattice", "far"])
def test_sets_of_any_k(gpu, kind, layout):
    """k whose rows wrap across a wave's lanes, both widths of kept entries."""
    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree

    pos = _lattice(21) if kind == "lattice" else datagen.clustered(9011, 1.0, nhalo=9, seed=3)[0]
    pos = pos + 1e6 if kind == "far" else pos
    p = _dev(pos)
    tm = DeviceTree(p, kerntype=nb.KSPH, form=nb.FORM_MIXED)
    tp = DeviceTree(p, kerntype=nb.KSPH)
    for k in (1, 6, 7, 20, 32, 33, 50, 64):
        print(f"mixed routes sets {kind} layout={layout} k={k}", flush=True)
        with _runs_mixed():
            nn, _ = _rows(tm, k, layout, d2=False)
        assert (nn.sort(1).values == _rows(tp, k, layout)[0].sort(1).values).all()


# tree heights 0..9: nodes are tested eight at a time from heights 3 and 6 on
@pytest.mark.parametrize("n", [20, 33, 65, 129, 256, 257, 1000, 2048, 2049, 4097, 9000])
@pytest.mark.parametrize("k", [8, 32, 33, 64])
def test_phase_by_tree_height(gpu, n, k):
    import torch

    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree

    k = min(k, n - 2)
    print(f"mixed routes phase n={n} k={k}", flush=True)
    x, v, _ = datagen.clustered(n, 1.0, nhalo=4, seed=n, with_vel=True)
    x, v = _dev(x), _dev(v / v.std())
    m = torch.tensor(datagen.lognormal_masses(n, n), device="cuda")
    t, p = (DeviceTree(x, mass=m, vel=v, treetype=nb.TPHS, aniso=-1, kerntype=nb.KSPH, form=f)
            for f in (nb.FORM_MIXED, nb.FORM_PLAIN))
    nn = torch.empty((n, k), dtype=torch.int32, device="cuda")
    rho, h, rp, hp = (torch.empty(n, dtype=torch.float64, device="cuda") for _ in range(4))
    with _runs_mixed():
        t.knn_density(k, nn, rho, h)
    p.density(k, rp, hp)
    assert torch.equal(nn.sort(1).values, _rows(p, k, nb.LAYOUT_BY_SLOT)[0].sort(1).values)
    assert torch.equal(h, hp)
    assert float((rho / rp - 1.0).abs().max()) < 1e-12
    with _runs_mixed():
        nn, _ = _rows(t, k, nb.LAYOUT_BY_ID, d2=False)
    assert torch.equal(nn.sort(1).values, _rows(p, k, nb.LAYOUT_BY_ID)[0].sort(1).values)


# A wave's queries are split among up to 32 waves, whose shares of a density
# cross between them; 131137: whole waves.  The reference sums the same lists
# with the kernel's own expression for a share, so only the order of some
# hundreds of positive terms differs: 300 roundings of 1.1e-16.  (Against the
# FP64 form's table lookup a particle with every neighbour at the edge of its
# kernel, k = 2, differs by 1e-11 of a density near 0.)
@pytest.mark.parametrize("n", [63, 65, 2049, 16385, 131137])
@pytest.mark.parametrize("k", [2, 31, 33])
def test_split_wave_densities(gpu, n, k):
    import torch

    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree

    print(f"mixed routes split waves n={n} k={k}", flush=True)
    p = _dev(datagen.clustered(n, 1.0, nhalo=5, seed=n)[0] if n > 100 else datagen.uniform(n, 1.0, n))
    m = torch.tensor(datagen.lognormal_masses(n, n), device="cuda")
    t = DeviceTree(p, mass=m, kerntype=nb.KSPH, form=nb.FORM_MIXED)
    nn = torch.empty((n, k), dtype=torch.int32, device="cuda")
    rho, h = (torch.empty(n, dtype=torch.float64, device="cuda") for _ in range(2))
    with _runs_mixed():
        t.knn_density(k, nn, rho, h)
    order, nn = t.order().long(), nn.long()
    x, ms = p[:, order], m[order]
    d2 = torch.zeros_like(nn, dtype=torch.float64)
    for c in range(3):
        d = x[c][:, None] - x[c][nn]
        d2 += d * d
    hs = 0.5 * d2.max(1).values.sqrt()
    assert torch.equal(h[order], hs)
    tab = np.zeros(1000)
    assert nb.lib().nbx_tree_kernel(t._h, None, nb._p(tab), 1000) == 1000
    tab = torch.tensor(tab, device="cuda")
    f = d2.sqrt() / hs[:, None] * 499.5
    i = f.long().clamp(max=998)
    w = torch.where(f < 999.0, tab[i] + (tab[i + 1] - tab[i]) * (f - i), tab[999]) * 0.5 / hs[:, None] ** 3
    want = (w * ms[nn]).sum(1)
    want.index_add_(0, nn.reshape(-1), (w * ms[:, None]).reshape(-1))
    assert float((rho[order] / want - 1.0).abs().max()) < 1e-13


def test_captured_search_with_scratch(gpu):
    """A captured search that needs scratch (a query per lane: few entries,
    many queries) replays to the eager answer, with other such searches on the
    tree, on the same stream and on another, between the replays."""
    import torch

    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree

    n, k = 300007, 4
    print("captured search with scratch", flush=True)
    t = DeviceTree(_dev(datagen.clustered(n, 100.0, nhalo=60, seed=5)[0]), kerntype=nb.KSPH)
    want = _rows(t, k, nb.LAYOUT_BY_ID)
    want3 = _rows(t, 3, nb.LAYOUT_BY_ID)
    nn, d2 = torch.empty_like(want[0]), torch.empty_like(want[1])
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        t.knn(k, nn, d2, variant=3, layout=nb.LAYOUT_BY_ID)
    side = torch.cuda.Stream()
    for _ in range(4):
        nn.fill_(-5)
        d2.fill_(-1.0)
        g.replay()
        with torch.cuda.stream(side):
            got3 = torch.empty_like(want3[0])
            t.knn(3, got3, None, variant=3, layout=nb.LAYOUT_BY_ID)
        torch.cuda.synchronize()
        assert torch.equal(nn, want[0]) and torch.equal(d2, want[1])
        assert torch.equal(got3, want3[0])
        assert torch.equal(_rows(t, 2, nb.LAYOUT_BY_ID)[0], want3[0][:, :2])
