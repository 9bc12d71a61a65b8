"""Pairs left out as exactly zero against covariances so flat that the FP32
determinant of a pair's sum decides: where it comes out negative the dense sums
hold a NaN, however far apart the points are, and so does the call."""
import numpy as np
import pytest

import dugma_amd as dg
from dugma_amd import workloads as W

pytestmark = pytest.mark.gpu


def _det32(S):
    """The pair kernel's determinant: FP32 products and FMAs (an FP64 product of
    two FP32 numbers is exact)."""
    f = np.float32

    def fma(a, b, c):
        return f(np.float64(a) * np.float64(b) + np.float64(c))

    a11, a12, a13, a22, a23, a33 = (f(S[i, j]) for i, j in ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)))
    c11 = fma(a22, a33, -f(a23 * a23))
    c12 = fma(a13, a23, -f(a12 * a33))
    c13 = fma(a12, a23, -f(a13 * a22))
    return fma(a11, c11, fma(a12, c12, f(a13 * c13)))


@pytest.mark.parametrize("flat", [1e-2, 1e-4, 1e-9])
def test_far_pairs_of_flat_covariances(flat):
    rng = np.random.default_rng(5)
    seen = set()
    for _ in range(24):
        Q = W.random_rotation(rng, 180.0)
        C = (Q @ np.diag([1.0, 1.0, flat]) @ Q.T).astype(np.float32).astype(np.float64)
        C = 0.5 * (C + C.T)
        m2 = C[0, 0] * C[1, 1] - C[0, 1] ** 2
        if not (m2 > 0 and np.linalg.det(C) > 0):
            continue  # left out by the validity rule
        P = rng.normal(size=(3, 70))
        _, h = dg.init(P, np.tile(C, (1, 70)), P + 400.0, np.tile(C, (1, 70)))
        try:
            if h.energy_info()[:2] != (70, 70):
                continue
            s2 = 2.0 ** (2 * np.round(-0.5 * np.log2(np.trace(C) / 3)))  # the context's scale (exact)
            det = _det32(2.0 * C * s2)
            E, g = dg.energy_grad(h, np.eye(3), np.zeros(3))
        finally:
            dg.fr_m(h)
        if det == 0:
            continue
        seen.add(bool(det < 0))
        assert np.isnan(E) == (det < 0), (flat, det, E)
        if det > 0:
            assert E == 0.0 and not g.any()
    assert False in seen or flat < 1e-6
