"""The search with a wave per query at the edges of its tree walk (one leaf,
six levels, one more), of its kept entries and of its 32-bit merge keys
(distances that FP32 does not tell apart, underflows or almost overflows), and
the search with a lane per query that takes over for few kept entries over many
queries.  Rows equal the (d2, ID)-sorted brute force entry by entry: every
distance is the same sum of squares in the same order."""
import numpy as np
import pytest

from nbodylib_amd import datagen

pytestmark = pytest.mark.gpu


def _rows(q, pos, k, target):
    d = np.zeros((len(q), len(pos)))
    for c in range(pos.shape[1]):
        d += (q[:, c][:, None] - pos[:, c][None, :]) ** 2
    if target:
        d[d == 0.0] = np.inf
    ids = np.lexsort((np.broadcast_to(np.arange(len(pos)), d.shape), d), axis=1)[:, :k]
    return ids, np.take_along_axis(d, ids, 1)


# leaves of 32 in trees of 0, 1, 6, 7 and 12 levels, their last leaves partial
@pytest.mark.parametrize("k", [1, 3, 4, 33, 64, 65, 128])
@pytest.mark.parametrize("n", [130, 2048, 2049, 5001, 131073])
def test_depths(gpu, n, k):
    import nbodylib_amd as nb

    print(f"wave search n={n} k={k}", flush=True)
    pos = datagen.uniform(n, 1.0, n)
    t = nb.KDTree(pos, kerntype=nb.KSPH)
    sel = np.random.default_rng(k).permutation(n)[:61]
    ids, dd = _rows(pos[sel], pos, k, True)
    nn, d2 = t.FindNearestTargets(sel.astype(np.int32), k)
    assert np.array_equal(d2, dd) and np.array_equal(nn, ids)
    nn, d2 = t.FindNearest(k)
    assert np.array_equal(d2[sel], dd) and np.array_equal(nn[sel], ids)


@pytest.mark.parametrize("n", [1, 2, 31, 33])
def test_few_particles(gpu, n):
    """Fewer particles than are kept: missing entries are -1 at 1e32."""
    import nbodylib_amd as nb

    print(f"wave search of {n} particles", flush=True)
    pos = datagen.uniform(n, 1.0, n)
    nn, d2 = nb.KDTree(pos, kerntype=nb.KSPH).FindNearestPosPoints(pos, 64)
    ids, dd = _rows(pos, pos, 64, False)
    assert np.array_equal(d2[:, :n], dd) and np.array_equal(nn[:, :n], ids)
    assert np.all(nn[:, n:] == -1) and np.all(d2[:, n:] == 1e32)


@pytest.mark.parametrize("scale", [1e-30, 1.0, 1e14])
@pytest.mark.parametrize("k", [5, 40, 64, 100])
def test_short_keys(gpu, k, scale):
    """Shells a few units in the last place thick around the query, among
    others well apart."""
    import nbodylib_amd as nb

    print(f"close distances k={k} scale={scale:g}", flush=True)
    r = np.random.default_rng(k)
    u = r.standard_normal((700, 3))
    u /= np.sqrt((u * u).sum(1))[:, None]
    radius = np.repeat([0.5, 0.75, 1.0], [30, 40, 630]) * (1.0 + 2.0**-50 * r.integers(0, 6, 700))
    radius[600:] *= r.uniform(0.1, 2.0, 100)
    pos = u * radius[:, None] * scale
    q = np.concatenate([np.zeros((1, 3)), pos[::97]])
    nn, d2 = nb.KDTree(pos, kerntype=nb.KSPH).FindNearestPosPoints(q, k)
    ids, dd = _rows(q, pos, k, False)
    assert np.array_equal(d2, dd) and np.array_equal(nn, ids)


@pytest.mark.parametrize("n", [40, 2049, 70000])
def test_phase_rows(gpu, n):
    import nbodylib_amd as nb

    print(f"6-D wave search n={n}", flush=True)
    r = np.random.default_rng(n)
    x = np.round(r.uniform(-1, 1, (n, 6)), 1 if n < 3000 else 3)  # many equal distances
    t = nb.KDTree(np.ascontiguousarray(x[:, :3]), vel=np.ascontiguousarray(x[:, 3:]), treetype=nb.TPHS, aniso=-1,
                  kerntype=nb.KSPH)
    for k in (1, 33, 64):
        k = min(k, n // 2)
        nn, d2 = t.FindNearestPhase(k)
        sel = r.permutation(n)[:40]
        ids, dd = _rows(x[sel], x, k, True)
        ok = dd < np.inf
        assert np.array_equal(d2[sel][ok], dd[ok]) and np.array_equal(nn[sel][ok], ids[ok])


@pytest.mark.parametrize("k", [1, 4, 5, 12, 13, 17, 18])
@pytest.mark.parametrize("kind", ["clustered", "lattice"])
def test_lane_per_query(gpu, kind, k):
    """Past 606208 queries (fewer for fewer entries) at most 18 kept entries are
    searched with a lane per query; a list of the same particles still runs with
    a wave per query."""
    import torch
    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree

    ax = np.arange(85.0)
    if kind == "lattice":
        pos = np.stack(np.meshgrid(ax, ax, ax, indexing="ij"), -1).reshape(-1, 3)
        pos = pos[np.random.default_rng(1).permutation(len(pos))]
    else:
        pos = datagen.clustered(606208 + 37, 1.0, nhalo=60, seed=5)[0]
    n = len(pos)
    print(f"lane per query {kind} n={n} k={k}", flush=True)
    period = 85.0 if kind == "lattice" else 1.0
    t = nb.KDTree(pos, kerntype=nb.KSPH, period=period)
    every = np.arange(n, dtype=np.int32)
    for per in (False, True):
        if per and k == 18:
            continue  # (19 kept entries)
        nn, d2 = t.FindNearest(k) if per else t.FindNearestNonPeriodic(k)
        wn, wd = t.FindNearestTargets(every, k, variant=nb.KNN_FINDNEAREST if per else nb.KNN_NONPERIODIC)
        assert np.array_equal(d2, wd) and np.array_equal(nn, wn)
    # densities of the same neighbours (in h and in the sums both are FP64)
    dev = torch.from_numpy(np.ascontiguousarray(pos.T)).cuda()
    rho, h = (torch.empty(n, device="cuda", dtype=torch.float64) for _ in range(2))
    if k > 1:
        DeviceTree(dev, kerntype=nb.KSPH).density(k, rho, h, variant=1)
        nn, d2 = t.FindNearestNonPeriodic(k)
        hh = 0.5 * np.sqrt(d2[:, -1])
        assert np.allclose(h.cpu().numpy(), hh, rtol=1e-15, atol=0)
        w = np.sqrt(d2) / hh[:, None]
        kern = np.where(w < 1, 1 - 0.75 * (2 - w) * w * w, 0.25 * np.clip(2 - w, 0, None) ** 3) / np.pi
        want = (kern / hh[:, None] ** 3 / n).sum(1)
        # the table's linear steps: at most W'' (2/999)^2 / 8 per entry, W'' <= 3 / pi
        err = k * (3 / np.pi) * (2 / 999) ** 2 / 8 / hh**3 / n
        assert np.all(np.abs(rho.cpu().numpy() - want) <= 1.5 * err)
