"""Work memory of the differentiation form over a stored list: no more than a
call uses, none for the smallest ones, and where there is no room for it the
kernels that need none give the same results."""
import numpy as np
import pytest

from nbodylib_amd import datagen

pytestmark = pytest.mark.gpu


def _set(n, k, shuffled=False):
    import torch

    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree

    p = torch.tensor(datagen.clustered(n, 1.0, nhalo=5, seed=n)[0].T.copy(), device="cuda")
    m = torch.tensor(datagen.lognormal_masses(n, n), device="cuda")
    t = DeviceTree(p, mass=m, kerntype=nb.KSPH)
    nn = torch.empty((n, k), dtype=torch.int32, device="cuda")
    d2 = torch.empty((n, k), dtype=torch.float64, device="cuda")
    t.knn(k, nn, d2, variant=nb.KNN_NONPERIODIC, layout=nb.LAYOUT_BY_ID if shuffled else nb.LAYOUT_BY_SLOT)
    if not shuffled:
        o = t.order().long()
        p, m = p[:, o].contiguous(), m[o].contiguous()
    del t, d2
    return p, m, nn


def _peak(f):
    """Most bytes of torch's that f held beyond what it found."""
    import torch

    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = f()
    torch.cuda.synchronize()
    return torch.cuda.max_memory_allocated() - before, out


def test_forward_memory(gpu):
    """Records and ranks, 36 bytes a particle, beside the two outputs."""
    from nbodylib_amd.device import sph_density

    n, k = 500000, 12
    print(f"sph work n={n} k={k}", flush=True)
    p, m, nn = _set(n, k)
    got, _ = _peak(lambda: sph_density(p, m, nn))
    assert got < (16 + 40) * n


@pytest.mark.parametrize("refused", [0, 1300000])  # work memory of every pass, or the backward's, which is larger
@pytest.mark.parametrize("shuffled", [False, True])
def test_no_room(gpu, monkeypatch, shuffled, refused):
    import torch

    from nbodylib_amd.device import SPHDensity, sph_density

    n, k = 20000, 12
    print(f"sph without work memory n={n} k={k} shuffled={shuffled} refused from {refused}", flush=True)
    p, m, nn = _set(n, k, shuffled)

    def run():
        rho, h = sph_density(p, m, nn)
        pg, mg = p.clone().requires_grad_(), m.clone().requires_grad_()
        r = SPHDensity.apply(pg, mg, nn)
        r.backward(1.0 / r.detach())
        return rho, h, r.detach(), pg.grad, mg.grad

    want = run()
    real, sizes = torch.empty, []

    def full(*size, **kw):
        if kw.get("dtype") == torch.uint8:
            sizes.append(size[0])
            if size[0] >= refused:
                raise torch.OutOfMemoryError("no room")
        return real(*size, **kw)

    monkeypatch.setattr(torch, "empty", full)
    got = run()
    monkeypatch.undo()
    assert len(sizes) == 3 and max(sizes) >= refused and (min(sizes) < refused) == (refused > 0)
    assert torch.equal(got[1], want[1])
    for a, b in zip(got, want):
        assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())
    assert float((got[0] / want[0] - 1.0).abs().max()) < 1e-12


@pytest.mark.parametrize("n,k", [(5, 4), (100, 32), (256, 32), (1024, 8), (257, 32), (1025, 8)])
def test_small_lists(gpu, n, k):
    """Up to 8192 entries no work memory, and the packed kernels' results."""
    import torch

    import nbodylib_amd as nb
    from nbodylib_amd.device import _check, _ptr, _stream, lib, sph_density

    print(f"sph small n={n} k={k}", flush=True)
    p = torch.tensor(datagen.uniform(n, 1.0, n).T.copy(), device="cuda")
    m = torch.tensor(datagen.lognormal_masses(n, n), device="cuda")
    # no particle in its own row: as the last entry it would make h zero
    rows = [(i + 1 + np.random.default_rng(i).permutation(n - 1)[:k]) % n for i in range(n)]
    nn = torch.tensor(np.stack(rows).astype(np.int32), device="cuda")
    held, (rho, h) = _peak(lambda: sph_density(p, m, nn))
    out = 2 * ((8 * n + 511) // 512 * 512)  # (blocks of 512 bytes)
    assert (held <= out) == (n * k <= 8192)
    w = torch.empty(lib().nbx_sph_work_bytes(n), dtype=torch.uint8, device="cuda")
    r2, h2 = torch.empty_like(rho), torch.empty_like(h)
    _check(lib().nbx_sph_density_fwd_ordered_dev(_ptr(p), _ptr(m), _ptr(nn), None, n, k, _ptr(r2), _ptr(h2), _ptr(w),
                                                 _stream()))
    assert torch.equal(h, h2)
    assert float((rho - r2).abs().max()) <= 1e-12 * float(r2.abs().max())
