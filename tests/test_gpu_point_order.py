"""Query points in any order: rows belong to the caller's points, for counts
around a wave, points outside the box and coinciding points, in 3-D and in
phase space."""
import numpy as np
import pytest

import oracle
from nbodylib_amd import datagen

pytestmark = pytest.mark.gpu


def _points(m, seed):
    rng = np.random.default_rng(seed)
    q = rng.uniform(-0.3, 1.3, (m, 3))
    q[::7] = q[0]          # coinciding points share a key
    q[1::11, 1] = 5.0      # far outside: the border cells
    return q


@pytest.mark.parametrize("m", [1, 64, 65, 129, 1000])
def test_rows_belong_to_their_points(gpu, m):
    import nbodylib_amd as nb

    n, k = 3000, 12
    print(f"point order m={m}", flush=True)
    pos, _ = datagen.clustered(n, 1.0, nhalo=5, seed=m)
    q = _points(m, m + 1)
    t = nb.KDTree(pos, kerntype=nb.KSPH)
    nn, d2 = t.FindNearestPosPoints(q, k)
    oi, od = oracle.Tree(pos, b=16).knn_points(q, k)
    assert np.array_equal(d2, od) and np.array_equal(np.sort(nn, 1), np.sort(oi, 1))
    w = np.random.default_rng(m + 2).random(n)
    mean = t.CalcSmoothLocalMeanPosition(q, w, k, rho=np.ones(n))
    one = np.array([t.CalcSmoothLocalMeanPosition(q[i:i + 1], w, k, rho=np.ones(n))[0] for i in (0, m // 2, m - 1)])
    # same kernels and row order one at a time: the sums agree to their rounding (k terms)
    assert np.allclose(mean[[0, m // 2, m - 1]], one, rtol=1e-13, atol=0)


@pytest.mark.parametrize("m", [64, 65, 200])
def test_phase_rows_belong_to_their_points(gpu, m):
    import nbodylib_amd as nb

    n, k = 2500, 9
    print(f"phase point order m={m}", flush=True)
    x, v, _ = datagen.clustered(n, 1.0, nhalo=4, seed=m, with_vel=True)
    v = v / v.std()
    t = nb.KDTree(x, vel=v, treetype=nb.TPHS, aniso=-1, kerntype=nb.KSPH)
    q, qv = _points(m, m + 3), 3.0 * _points(m, m + 4)
    nn, d2 = t.FindNearestPhasePoints(q, qv, k)
    d = np.zeros((m, n))
    for a, b in ((q, x), (qv, v)):
        for c in range(3):
            d += (a[:, c][:, None] - b[:, c][None, :]) ** 2
    assert np.array_equal(d2, np.sort(d, 1)[:, :k])
    assert np.array_equal(np.take_along_axis(d, nn.astype(np.int64), 1), d2)
