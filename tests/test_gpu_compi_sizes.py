"""compi at sizes around its 64-target sub-tiles, its 8- and 32-source moment
blocks and the source count where the latter change, against the oracle."""
import numpy as np
import pytest

import dugma_amd as dg
from dugma_amd import workloads as W
from test_gpu_compi import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(1, 1), (63, 7), (64, 8), (65, 9), (257, 31), (130, 33), (300, 100)])
def test_sizes(oracle, n, m):
    # variances of its own: the workloads' come from 8 neighbours, which the
    # smallest of these clouds do not have
    rng = np.random.default_rng(1000 * n + m)
    d = dict(X=rng.random((3, n)), X_C=W.iso_blocks(rng.uniform(0.01, 0.05, n)), Y=rng.random((3, m)),
             Y_C=W.iso_blocks(rng.uniform(0.01, 0.05, m)))
    check(oracle, d, W.random_rotation(rng, 5.0), np.array([0.01, -0.02, 0.005]), 0.7)


def test_source_blocks_agree():
    """Beyond 65,536 sources the moments are summed over 32 a workgroup: the
    coefficients are sums over sources, so those of the whole cloud are the
    halves' added (FP64 sums of FP32 weights, the same ones up to the FP32
    sub-tiles, which the source split does not change)."""
    rng = np.random.default_rng(2)
    n, m = 64, 65600
    X, Y = rng.random((3, n)), rng.random((3, m))
    CX, CY = W.iso_blocks(np.full(n, 0.02)), W.iso_blocks(np.full(m, 0.03))
    R, t = W.random_rotation(rng, 5.0), np.array([0.01, -0.02, 0.005])

    def coef(sl):
        _, h = dg.init(X, CX, Y[:, sl], CY[:, 3 * sl.start:3 * sl.stop])
        try:
            return dg.compi(h, R, t, sig=0.8)
        finally:
            dg.fr_m(h)

    whole = coef(slice(0, m))
    parts = coef(slice(0, 30000)) + coef(slice(30000, m))
    assert np.abs(whole - parts).max() <= 1e-12 * np.abs(whole).max()
