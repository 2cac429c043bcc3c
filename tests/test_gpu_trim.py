"""Device memory kept by the library goes back to the device on request."""
import pytest

from nbodylib_amd import datagen

pytestmark = pytest.mark.gpu


def test_trim_memory(gpu):
    import torch

    import nbodylib_amd as nb

    n = 400000
    print(f"trim memory n={n}", flush=True)
    pos = datagen.uniform(n, 1.0, 3)
    want = nb.KDTree(pos, kerntype=nb.KSPH).FindNearest(8)
    nb.trim_memory()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    got = nb.KDTree(pos, kerntype=nb.KSPH).FindNearest(8)
    held = free - torch.cuda.mem_get_info()[0]
    assert held > 0 and nb.trim_memory() >= held // 2
    assert torch.cuda.mem_get_info()[0] >= free - (2 << 20)
    assert nb.trim_memory() == 0
    assert (got[0] == want[0]).all() and (got[1] == want[1]).all()
    assert (nb.KDTree(pos, kerntype=nb.KSPH).FindNearest(8)[0] == want[0]).all()
