"""Small sets split the queries of a wave among several waves in the precision
form's own kernel (rows in key order): rows against the exact ones as sets, in
ascending order up to the keys' resolution, and the symmetric density, whose
shares cross the parts, against FP64."""
import numpy as np
import pytest

from nbodylib_amd import datagen

pytestmark = pytest.mark.gpu


# waves: 1, 2, 33, 64, 257 and around the 2048 from which on waves are whole
@pytest.mark.parametrize("k", [2, 31, 33])
@pytest.mark.parametrize("n", [63, 65, 2049, 4096, 16385, 131072, 131137])
def test_parts(gpu, n, k):
    import torch
    import nbodylib_amd as nb
    from nbodylib_amd.device import DeviceTree

    print(f"split waves n={n} k={k}", flush=True)
    pos = datagen.clustered(n, 1.0, nhalo=5, seed=n)[0] if n > 100 else datagen.uniform(n, 1.0, n)
    dev = torch.from_numpy(np.ascontiguousarray(pos.T)).cuda()
    t = DeviceTree(dev, kerntype=nb.KSPH, form=nb.FORM_MIXED)
    nn = torch.empty((n, k), device="cuda", dtype=torch.int32)
    rho, h, rp, hp = (torch.empty(n, device="cuda", dtype=torch.float64) for _ in range(4))
    t.knn_density(k, nn, rho, h)
    p = DeviceTree(dev, kerntype=nb.KSPH, form=nb.FORM_PLAIN)
    en = torch.empty_like(nn)
    d2 = torch.empty((n, k), device="cuda", dtype=torch.float64)
    p.knn(k, en, d2, variant=nb.KNN_NONPERIODIC, layout=nb.LAYOUT_BY_SLOT)
    assert torch.equal(torch.sort(nn, 1).values, torch.sort(en, 1).values)
    x = dev[:, t.order().long()]
    d = ((x[:, :, None] - x[:, nn.long()]) ** 2).sum(0)
    # keys: FP32 distances short of their last 6 (k > 32: 4) bits, and the
    # offsets' roundings, which a leaf's size scales
    assert torch.all(d[:, 1:] >= d[:, :-1] * (1 - 2.0**-14) - 2.0**-20 * d[:, -1:])
    p.density(k, rp, hp)
    assert torch.equal(h, hp)
    assert float((rho / rp - 1.0).abs().max()) < 2e-6
