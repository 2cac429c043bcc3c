"""Searches at the edges of their kept-entry groups (33, 65 and 129 entries) and
where ties cross the k-th distance: rows equal the (d2, ID)-sorted brute force
entry by entry.  The forward density summed in the search equals the one over
the same lists."""
import numpy as np
import pytest

import oracle
from nbodylib_amd import datagen

pytestmark = pytest.mark.gpu

KS = [1, 2, 31, 32, 33, 34, 64, 65, 66, 128, 129]


def _rows(q, pos, k, target):
    """(d2, ID)-sorted rows; target: d2 == 0 is no neighbour."""
    d = np.zeros((len(q), len(pos)))
    for c in range(3):
        d += (q[:, c][:, None] - pos[:, c][None, :]) ** 2
    if target:
        d[d == 0.0] = np.inf
    ids = np.lexsort((np.broadcast_to(np.arange(len(pos)), d.shape), d), axis=1)[:, :k]
    return ids, np.take_along_axis(d, ids, 1)


def _lattice(g):
    ax = np.arange(g) + 0.5
    p = np.stack(np.meshgrid(ax, ax, ax, indexing="ij"), -1).reshape(-1, 3)
    return p[np.random.default_rng(g).permutation(len(p))]  # IDs in no spatial order


@pytest.mark.parametrize("k", KS)
@pytest.mark.parametrize("kind", ["clustered", "lattice"])
@pytest.mark.parametrize("form", ["plain", "mixed"])
def test_rows_exact(gpu, form, kind, k):
    import nbodylib_amd as nb

    pos = _lattice(9) if kind == "lattice" else datagen.clustered(911, 1.0, nhalo=4, seed=5)[0]
    print(f"kept entries {form} {kind} n={len(pos)} k={k}", flush=True)
    t = nb.KDTree(pos, kerntype=nb.KSPH, form=nb.FORM_PLAIN if form == "plain" else nb.FORM_MIXED)
    nn, d2 = t.FindNearest(k)
    ids, dd = _rows(pos, pos, k, True)
    assert np.array_equal(d2, dd) and np.array_equal(nn, ids)
    if form == "mixed":  # by slot: the same rows through the tree order
        order = t.order()
        ns, ds = t.FindNearest(k, layout=nb.LAYOUT_BY_SLOT)
        assert np.array_equal(ds, dd[order]) and np.array_equal(order[ns], ids[order])
        return
    # positions: particles (found at d2 = 0), lattice cell centres, far outside
    q = np.concatenate([pos[:70], pos[:40] + 0.5, pos[:5] + 1e3])
    nn, d2 = t.FindNearestPosPoints(q, k)
    ids, dd = _rows(q, pos, k, False)
    assert np.array_equal(d2, dd) and np.array_equal(nn, ids)


@pytest.mark.parametrize("k", [6, 7, 32, 64, 128])
def test_periodic_lattice(gpu, k):
    import nbodylib_amd as nb

    pos = _lattice(8)
    print(f"periodic lattice k={k}", flush=True)
    t = nb.KDTree(pos, kerntype=nb.KSPH, period=8.0)
    nn, d2 = t.FindNearest(k)
    bi, bd = oracle.knn_brute(pos, k, mode=1, period=8.0)
    assert np.array_equal(d2, bd) and np.array_equal(np.sort(nn, 1), np.sort(bi, 1))


def test_coinciding_particles(gpu):
    """More particles at one point than are kept: the smallest IDs stay, and a
    target search, which skips them all, reports the others."""
    import nbodylib_amd as nb

    rng = np.random.default_rng(8)
    pos = rng.random((600, 3))
    pos[rng.permutation(600)[:90]] = 0.25
    t = nb.KDTree(pos, kerntype=nb.KSPH)
    q = np.concatenate([np.full((3, 3), 0.25), pos[:66]])
    for k in (20, 40):
        print(f"coinciding k={k}", flush=True)
        nn, d2 = t.FindNearestPosPoints(q, k)
        ids, dd = _rows(q, pos, k, False)
        assert np.array_equal(d2, dd) and np.array_equal(nn, ids)
        nn, d2 = t.FindNearest(k)
        ids, dd = _rows(pos, pos, k, True)
        assert np.array_equal(d2, dd) and np.array_equal(nn, ids)


@pytest.mark.parametrize("k", [2, 31, 32, 33, 64, 65, 129])
@pytest.mark.parametrize("form", ["plain", "mixed"])
def test_forward_in_search(gpu, form, k):
    """Sums of k own and as many scattered terms as a particle is a neighbour
    to: a few hundred roundings of 1.1e-16 each, in any order."""
    import torch

    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree, sph_density

    n = 1500
    print(f"forward in search {form} k={k}", flush=True)
    pos = torch.tensor(datagen.clustered(n, 1.0, nhalo=5, seed=k)[0].T.copy(), device="cuda")
    m = torch.tensor(datagen.lognormal_masses(n, k), device="cuda")
    t = DeviceTree(pos, mass=m, kerntype=nb.KSPH, form=nb.FORM_PLAIN if form == "plain" else nb.FORM_MIXED)
    nn = torch.empty((n, k), dtype=torch.int32, device="cuda")
    d2 = torch.empty((n, k), dtype=torch.float64, device="cuda")
    t.knn(k, nn, d2, layout=nb.LAYOUT_BY_ID)
    ro, ho = sph_density(pos, m, nn)
    rho, h = torch.empty_like(ro), torch.empty_like(ho)
    t.sph_density(k, rho, h, block_rows=1024)
    assert torch.equal(h, ho)
    assert float((rho / ro - 1.0).abs().max()) < 1e-12


@pytest.mark.parametrize("n", [20, 33, 65, 129, 256, 257, 1000, 2048, 2049, 4097, 9000])
@pytest.mark.parametrize("k", [8, 32, 64])
def test_phase_rows_by_tree_height(gpu, n, k):
    """6-D precision form: trees below, at and above the heights (3 and 6) from
    which nodes are tested eight at a time."""
    import nbodylib_amd as nb

    k = min(k, n - 2)
    print(f"phase rows n={n} k={k}", flush=True)
    x, v, _ = datagen.clustered(n, 1.0, nhalo=4, seed=n, with_vel=True)
    v = v / v.std()
    t = nb.KDTree(x, vel=v, treetype=nb.TPHS, aniso=-1, kerntype=nb.KSPH, form=nb.FORM_MIXED)
    nn, d2 = t.FindNearestPhase(k)
    ph = np.concatenate([x, v], 1)
    for a in range(0, n, 1500):
        d = np.zeros((len(ph[a:a + 1500]), n))
        for c in range(6):
            d += (ph[a:a + 1500, c][:, None] - ph[:, c][None, :]) ** 2
        d[d == 0.0] = np.inf
        assert np.array_equal(d2[a:a + 1500], np.sort(d, 1)[:, :k])
        assert np.array_equal(np.take_along_axis(d, nn[a:a + 1500].astype(np.int64), 1), d2[a:a + 1500])
