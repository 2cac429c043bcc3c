"""FOF's walk opens six levels at a time from the root: trees below, at and
above those heights, linking lengths from a few pairs to everything joined,
against all pairs; and sets where many particles share one group, where links
are joined a candidate per lane."""
import numpy as np
import pytest

import oracle
from nbodylib_amd import datagen

pytestmark = pytest.mark.gpu

# leaves: 1, 2, 3, 33, 64, 65, 129 (a level of 64 leaves is 2048 particles)
SIZES = [20, 33, 64, 65, 1050, 2048, 2049, 4100]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("kind", ["uniform", "clustered"])
@pytest.mark.parametrize("periodic", [False, True])
def test_levels(gpu, n, kind, periodic):
    import nbodylib_amd as nb

    pos = datagen.uniform(n, 1.0, n) if kind == "uniform" else datagen.clustered(n, 1.0, nhalo=3, seed=n)[0]
    per = 1.0 if periodic and n > 16 else None
    t = nb.KDTree(pos, kerntype=nb.KSPH, period=per)
    for f in (0.05, 0.3, 0.7, 1.0, 3.0, 20.0):
        b = f * datagen.mean_spacing(n, 1.0)
        if per is not None and b >= 0.5:
            continue
        print(f"fof levels {kind} n={n} periodic={periodic} b={f} spacings", flush=True)
        for minnum in (1, 2, 8):
            lab, ng = t.FOF(b, minnum)
            ol, og = oracle.fof_brute(pos, b, minnum, period=per)
            assert ng == og and np.array_equal(lab, ol)


@pytest.mark.parametrize("n", SIZES)
def test_levels_phase(gpu, n):
    import nbodylib_amd as nb

    x, v, _ = datagen.clustered(n, 1.0, nhalo=3, seed=n + 1, with_vel=True)
    v = 0.2 * v / v.std()
    t = nb.KDTree(x, vel=v, treetype=nb.TPHS, aniso=-1, kerntype=nb.KSPH)
    for b in (0.02, 0.1, 0.3, 3.0):
        print(f"fof levels phase n={n} b={b}", flush=True)
        lab, ng = t.FOF(b, 2)
        ol, og = oracle.fof_brute(x, b, 2, vel=v)
        assert ng == og and np.array_equal(lab, ol)
        s = b * b
        lab, ng = t.FOFCriterion(nb.FOF_CMP_6D, [nb.TPHS, s, s, 0, 0, 0, s, s], 2)
        assert ng == og and np.array_equal(lab, ol)


@pytest.mark.parametrize("n", [70001, 140000])
def test_deeper_trees(gpu, n):
    import nbodylib_amd as nb

    pos = datagen.clustered(n, 100.0, nhalo=40, seed=n)[0]
    t = nb.KDTree(pos, kerntype=nb.KSPH, period=100.0)
    ot = oracle.Tree(pos, b=16, kerntype=oracle.KSPH, period=100.0)
    for f in (0.2, 0.6):
        b = f * datagen.mean_spacing(n, 100.0)
        print(f"fof deeper n={n} b={f} spacings", flush=True)
        lab, ng = t.FOF(b, 5)
        raw, _ = ot.fof(b, 5)
        ol, og = oracle.fof_canonical(raw, 5)
        assert ng == og and np.array_equal(lab, ol)


@pytest.mark.parametrize("size", [2, 3, 12, 13, 70, 5000])
def test_group_sums(gpu, size):
    """Sizes and smallest IDs where a wave of 64 particles holds more groups
    than it sums, a few, and a part of one: n / size tight groups far apart."""
    import nbodylib_amd as nb

    n = 15000 // size * size
    print(f"group sums size={size} n={n}", flush=True)
    rng = np.random.default_rng(size)
    ng = n // size
    centre = np.stack(np.unravel_index(rng.permutation(8000)[:ng], (20, 20, 20)), -1).astype(float)
    group = rng.permutation(np.repeat(np.arange(ng), size))  # members of a group all over the IDs
    pos = centre[group] + rng.uniform(-0.01, 0.01, (n, 3))
    lab, got = nb.KDTree(pos, kerntype=nb.KSPH).FOF(0.1, 2)
    assert got == ng
    # equal sizes: numbered by smallest member
    first = np.full(ng, n)
    np.minimum.at(first, group, np.arange(n))
    want = np.empty(ng, dtype=np.int64)
    want[np.argsort(first)] = np.arange(1, ng + 1)
    assert np.array_equal(lab, want[group])
