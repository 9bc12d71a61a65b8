"""The pair passes leave out pairs whose FP32 term is exactly zero (spatial
index, csrc/dugma_near.h).  Against the FP64 oracle, which sums every pair, at
the sizes where the index can go wrong: single points, partial 64-point blocks
and sub-tiles, more streamed points than one window of bits holds, kernels that
reach every pair, kernels that reach almost none, clouds out of each other's
reach, and covariances stretched by an R that is not a rotation."""
import numpy as np
import pytest

import dugma_amd as dg
from dugma_amd import workloads as W

pytestmark = pytest.mark.gpu

E_TOL = 1e-6  # the library's own bars
G_TOL = 1e-5


def rel(a, b):
    a, b = np.asarray(a, float), np.asarray(b, float)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def f32(a):
    return np.asarray(a, np.float64).astype(np.float32).astype(np.float64)


def clouds(n, m, D, width, full, seed):
    """Points on a noisy unit circle / sphere with a few outliers; standard
    deviations about `width`, a factor 2 apart (full: random orientations)."""
    rng = np.random.default_rng(seed)

    def points(k):
        u = rng.normal(size=(k, D))
        u /= np.linalg.norm(u, axis=1, keepdims=True)
        u += rng.normal(scale=0.002, size=u.shape)
        out = rng.random(k) < 0.03
        u[out] *= rng.uniform(0.0, 3.0, size=(int(out.sum()), 1))
        return f32(u)

    def covs(k):
        s = width * rng.uniform(0.7, 1.4, size=(k, D if full else 1))
        if not full:
            return f32((s ** 2)[:, :, None] * np.eye(D))
        Q = np.linalg.qr(rng.normal(size=(k, D, D)))[0]
        C = np.einsum("nab,nb,ncb->nac", Q, s ** 2, Q)
        return f32(0.5 * (C + np.transpose(C, (0, 2, 1))))

    return points(n), covs(n), points(m), covs(m)


def rotation(D, deg=7.0):
    a = np.deg2rad(deg)
    return W.rot2(a) if D == 2 else W.rot_axis_angle([0.3, -0.5, 0.8], a)


def context(Y, SY, X, SX):
    return dg.init(Y.T.copy(), W.blocks(SY), X.T.copy(), W.blocks(SX))[1]


@pytest.mark.parametrize("full", [False, True], ids=["iso", "full"])
@pytest.mark.parametrize("width", [0.02, 3.0], ids=["narrow", "wide"])
@pytest.mark.parametrize("D,n,m", [(3, 1, 1), (3, 63, 65), (3, 64, 64), (3, 129, 1), (3, 1, 300), (3, 1500, 4097),
                                   (2, 65, 63), (2, 2100, 700)])
def test_all_pairs_against_the_oracle(oracle, D, n, m, width, full):
    Y, SY, X, SX = clouds(n, m, D, width, full, seed=n + 7 * m)
    X[0] = f32(rotation(D).T @ Y[0] + 0.3 * width)  # at least one pair in reach
    R, t = rotation(D), np.full(D, 0.01 * width)
    ref = oracle.energy(Y, SY, X, SX, R, t, grads=True)
    h = context(Y, SY, X, SX)
    try:
        E0 = dg.energy(h, R, t)
        E, g = dg.energy_grad(h, R, t)
        pts = dg.energy_grad_points(h, R, t)
        hess = dg.energy_grad_hess(h, R, t) if D == 3 else None
    finally:
        dg.fr_m(h)
    for e in (E0, E, pts["E"]) + ((hess[0],) if hess else ()):
        assert abs(e / ref["E"] - 1) <= E_TOL
    # against the gradient's own terms: a few pairs' torques may cancel
    scale = max(np.linalg.norm(ref["gpose"]), np.abs(ref["gY"]).sum())
    for gp in (g, pts["gpose"]) + ((hess[1],) if hess else ()):
        assert np.linalg.norm(gp - ref["gpose"]) <= G_TOL * scale
    for a, b in (("gX", "gY"), ("gXC", "gSY"), ("gY", "gX"), ("gYC", "gSX")):
        assert rel(pts[a], ref[b]) <= G_TOL, a


def test_more_streamed_points_than_one_window(oracle):
    """270,001 points stream past 70 in more than one window of 2^18 bits, in
    both roles (pose pass: the targets stream; per-point passes: both)."""
    Y, SY, X, SX = clouds(270001, 70, 3, 0.01, False, seed=5)
    R, t = rotation(3), np.zeros(3)
    ref = oracle.energy(Y, SY, X, SX, R, t, grads=True)
    for swap in (False, True):
        if swap:  # E is symmetric: the clouds exchanged under the inverse pose
            h, Rs = context(X, SX, Y, SY), R.T.copy()
        else:
            h, Rs = context(Y, SY, X, SX), R
        try:
            E, g, H = dg.energy_grad_hess(h, Rs, t)
            E2, g2 = dg.energy_grad(h, Rs, t)
            pts = dg.energy_grad_points(h, Rs, t)
        finally:
            dg.fr_m(h)
        for e in (E, E2, pts["E"]):
            assert abs(e / ref["E"] - 1) <= E_TOL
        assert rel(g, g2) <= 1e-12 and np.all(np.isfinite(H))
        if not swap:
            assert rel(g2, ref["gpose"]) <= G_TOL
            assert rel(pts["gX"], ref["gY"]) <= G_TOL and rel(pts["gYC"], ref["gSX"]) <= G_TOL


def test_clouds_out_of_reach_give_zero():
    Y, SY, X, SX = clouds(500, 400, 3, 0.02, True, seed=9)
    h = context(Y, SY, X, SX)
    try:
        E, g, H = dg.energy_grad_hess(h, np.eye(3), np.array([50.0, 0.0, 0.0]))
        pts = dg.energy_grad_points(h, np.eye(3), np.array([50.0, 0.0, 0.0]))
    finally:
        dg.fr_m(h)
    assert E == 0.0 and not g.any() and not H.any()
    assert pts["E"] == 0.0 and not any(pts[k].any() for k in ("gX", "gXC", "gY", "gYC", "gpose", "gdT"))


def test_pose_that_is_not_a_rotation(oracle):
    """R = 3 x a rotation stretches the source covariances (full records): the
    reach follows."""
    Y, SY, X, SX = clouds(900, 800, 3, 0.02, True, seed=11)
    Y = f32(3.0 * Y)
    R, t = 3.0 * rotation(3), np.zeros(3)
    ref = oracle.energy(Y, SY, X, SX, R, t, grads=True)
    h = context(Y, SY, X, SX)
    try:
        E, g = dg.energy_grad(h, R, t, cov="full")
        pts = dg.energy_grad_points(h, R, t)
    finally:
        dg.fr_m(h)
    assert abs(E / ref["E"] - 1) <= E_TOL and abs(pts["E"] / ref["E"] - 1) <= E_TOL
    assert rel(pts["gX"], ref["gY"]) <= G_TOL and rel(pts["gY"], ref["gX"]) <= G_TOL
