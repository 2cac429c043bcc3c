"""FOF around the size from which its linking kernel is persistent (twice the
waves that are resident at once: 655360 particles in 3-D, 524288 in 6-D)
against the oracle's tree: sets with few links, of one group per cell and of
dense halos, whose shares the waves of other XCDs drain."""
import numpy as np
import pytest

import oracle
from nbodylib_amd import datagen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [655297, 655361, 700001])
@pytest.mark.parametrize("kind,b", [("uniform", 0.2), ("uniform", 0.7), ("clustered", 0.2), ("halo", 0.2)])
def test_around_the_line(gpu, kind, b, n):
    import nbodylib_amd as nb

    print(f"fof forms {kind} n={n} b={b}", flush=True)
    if kind == "uniform":
        pos = datagen.uniform(n, 100.0, n)
    else:
        pos = datagen.clustered(n, 100.0, nhalo=150 if kind == "clustered" else 1, seed=n)[0]
    b *= datagen.mean_spacing(n, 100.0)
    raw, _ = oracle.Tree(pos, b=16, period=100.0).fof(b, 2)
    want, groups = oracle.fof_canonical(raw, 2)
    lab, ng = nb.KDTree(pos, kerntype=nb.KSPH, period=100.0).FOF(b, 2)
    assert ng == groups and np.array_equal(lab, want)


@pytest.mark.parametrize("n", [524225, 524353])
def test_around_the_line_phase(gpu, n):
    import nbodylib_amd as nb

    print(f"fof forms phase n={n}", flush=True)
    x, v, _ = datagen.clustered(n, 1.0, nhalo=150, seed=n, with_vel=True)
    v = 0.2 * v / v.std()
    b = 0.02
    raw, _ = oracle.Tree(x, vel=v, b=16, treetype=oracle.TPHS).fof(b, 4)
    want, groups = oracle.fof_canonical(raw, 4)
    t = nb.KDTree(x, vel=v, treetype=nb.TPHS, aniso=-1, kerntype=nb.KSPH)
    lab, ng = t.FOF(b, 4)
    assert groups > 0 and ng == groups and np.array_equal(lab, want)
    s = b * b
    lab, ng = t.FOFCriterion(nb.FOF_CMP_6D, [nb.TPHS, s, s, 0, 0, 0, s, s], 4)
    assert ng == groups and np.array_equal(lab, want)
