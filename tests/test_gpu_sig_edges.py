"""update_sig quantises the smallest squared distance of a chunk once: the same
value as the oracle, which quantises every pair, at the edges of the 8-candidate
steps and of the chunks, and with distances of 0, below the quantum, beyond the
u32 range and not finite."""
import numpy as np
import pytest

import dugma_amd as dg

pytestmark = pytest.mark.gpu


def _check(oracle, X, Y, R=None, t=None):
    D = X.shape[1]
    R = np.eye(D) if R is None else R
    t = np.zeros(D) if t is None else t
    C = np.tile(np.eye(D) * 0.01, (1, len(X)))
    CY = np.tile(np.eye(D) * 0.01, (1, len(Y)))
    _, h = dg.init(X.T, C, Y.T, CY)
    try:
        got = dg.update_sig(h, R, t)
    finally:
        dg.fr_m(h)
    ref = oracle.update_sig(X, Y, R, t)
    assert got == ref or (np.isnan(got) and np.isnan(ref)), (got, ref)


@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("n,m", [(1, 1), (3, 7), (64, 8), (65, 9), (257, 63), (256, 64), (255, 65), (1000, 1031),
                                 (31, 4099)])
def test_sizes(oracle, D, n, m):
    rng = np.random.default_rng(n * 10007 + m)
    _check(oracle, rng.normal(size=(n, D)), rng.normal(size=(m, D)))


@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("far", [0.0, 1e-5, 70.0, 1e4, 1e18, 1e25, np.inf, np.nan])
def test_values(oracle, D, far):
    """A few sources at distance `far` among ordinary ones, and alone."""
    rng = np.random.default_rng(7)
    X = rng.normal(size=(70, D))
    Y = rng.normal(size=(40, D))
    Y[[0, 8, 39]] = far
    with np.errstate(all="ignore"):
        _check(oracle, X, Y)
        _check(oracle, X, np.full((9, D), far))
