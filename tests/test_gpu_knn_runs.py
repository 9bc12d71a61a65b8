"""k-NN over a grid whose nearest cells are few or one: equal points, points on a
line along each axis, two distant clusters, against the oracle's brute force."""
import numpy as np
import pytest

import dugma_amd as dg
from dugma_amd import workloads as W

pytestmark = pytest.mark.gpu


def _cloud(kind, n, rng):
    if kind == "equal":
        return np.full((3, n), 0.5)
    if kind in "xyz":
        P = np.zeros((3, n))
        P["xyz".index(kind)] = rng.random(n)
        return P
    P = rng.normal(scale=0.01, size=(3, n))
    P[:, n // 3:] += 50.0
    return P


@pytest.mark.parametrize("k", [1, 8, 16, 32])
@pytest.mark.parametrize("kind", ["equal", "x", "y", "z", "clusters"])
def test_few_cells(oracle, kind, k):
    rng = np.random.default_rng(3)
    n, m = 4200, 4100  # above the all-pairs limit
    X, Y = _cloud(kind, n, rng), _cloud(kind, m, rng)
    _, h = dg.init(X, W.iso_blocks(np.full(n, 0.01)), Y, W.iso_blocks(np.full(m, 0.01)))
    try:
        R, t = np.eye(3), np.array([0.003, -0.001, 0.002])
        Xf, Yf = X.T.astype(np.float32), Y.T.astype(np.float32)
        idx, d2 = dg.knn(h, dg.KNN_TARGET_TO_SOURCE, k, R, t)
        ri, rd = oracle.knn(Xf, oracle.transform_points(Yf, R, t), k, False)
        np.testing.assert_array_equal(idx, ri)
        np.testing.assert_array_equal(d2, rd)
        idx, d2 = dg.knn(h, dg.KNN_SOURCE_SELF, k)
        ri, rd = oracle.knn(Yf, Yf, k, True)
        np.testing.assert_array_equal(idx, ri)
        np.testing.assert_array_equal(d2, rd)
    finally:
        dg.fr_m(h)
