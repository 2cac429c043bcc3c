"""Smoothed velocities, dispersions and moments at the edges of their blocks of
1024 rows, with row lengths that do and do not allow wide loads, and with
clusters whose shares cross the blocks; against the oracle, with the bounds of
the other comparisons (FP64 sums in another order: 1e-12 of the largest mean,
1e-11 of the largest dispersion, 1e-9 of the moments' quotients)."""
import numpy as np
import pytest

import oracle
from nbodylib_amd import datagen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [2, 5, 8, 33])
@pytest.mark.parametrize("n", [300, 1024, 1025, 2600])
def test_block_edges(gpu, n, k):
    import nbodylib_amd as nb

    print(f"smoothed velocities n={n} k={k}", flush=True)
    pos = datagen.clustered(n, 1.0, nhalo=3, seed=n)[0]
    vel = np.random.default_rng(n + k).standard_normal((n, 3))
    mass = np.random.default_rng(k).uniform(0.5, 2.0, n)
    order = np.random.default_rng(1).permutation(n)  # no leaf order in the IDs
    pos, vel = np.ascontiguousarray(pos[order]), np.ascontiguousarray(vel[order])
    t = nb.KDTree(pos, vel=vel, mass=mass, kerntype=nb.KSPH)
    ot = oracle.Tree(pos, vel=vel, mass=mass, b=16, kerntype=oracle.KSPH)
    om, od = ot.smooth_vel(k, disp=True)
    m, d = t.CalcSmoothVelDisp(k)
    assert np.max(np.abs(m - om)) < 1e-12 * np.max(np.abs(om))
    assert np.max(np.abs(d - od)) < 1e-11 * np.max(np.abs(od))
    if k < 5:
        return  # (dispersions of a particle or two vanish)
    osk, oku = ot.smooth_moments(k, om, od)
    sk, ku = t.CalcSmoothVelMoments(k, mean=om, disp=od)
    assert np.max(np.abs(sk - osk)) < 1e-9 * np.max(np.abs(osk))
    assert np.max(np.abs(ku - oku)) < 1e-9 * np.max(np.abs(oku))
