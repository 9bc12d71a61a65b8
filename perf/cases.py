"""What is measured of this library: calls that a registration program makes.

Every case goes through the Python mirror of the C ABI (`dugma_amd`).  The
clouds are the repository's own synthetic workloads (`dugma_amd.workloads`:
closed surfaces, structured-light clouds with outliers, depth views, 2-D
contours, Kinect-sized clouds, batched trials), from the smallest calls to the
200,000 x 200,000 one.  Coordinates and variances are single-precision values, as
a sensor's files hold them (the library's own state is FP32), so that `exact`
computes on the very same numbers.

`exact` is plain torch in 64 bits: dense all-pairs sums, a brute-force k-NN.
"""
import math

import numpy as np
import torch

import dugma_amd as dg
from dugma_amd import workloads as W


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # 2-D contours: one gradient evaluation of a small planar registration
        # (launches and latency)
        dict(name="contour_2d_1k", kind="pose", cloud="contour", n=1201, m=1000),
        # the smallest 3-D clouds, isotropic sigma: an optimiser's inner call
        dict(name="pose_iso_1k", kind="pose", cloud="iso", n=1000, m=1000),
        # structured-light clouds with full covariances and 10% outliers: the
        # gradient callback at the size the reference recommends
        dict(name="pose_full_6k", kind="pose", cloud="camera", n=6000, m=6000),
        # the large single pair: energy and pose gradient of one pose
        dict(name="pose_iso_200k", kind="pose", cloud="iso", n=200000, m=200000),
        # a Newton step of the energy registration: energy, gradient, Hessian
        dict(name="hess_iso_50k", kind="hess", cloud="iso", n=50021, m=47111),
        # gradients for every point and covariance of two 320 x 240 depth views
        dict(name="points_views_77k", kind="points", cloud="views", n=320, m=240),
        # one outer iteration with surface covariances: both clouds' covariance
        # update from the 8 nearest neighbours, then the gradient on them
        dict(name="iteration_surface_60k", kind="cov_iteration", cloud="iso", n=60001, m=49999),
        # the same with per-point sigma, at the large size
        dict(name="iteration_sigma_200k", kind="sigma_iteration", cloud="iso", n=200000, m=200000),
        # the reference's own two GPU calls at the size it recommends
        dict(name="update_sig_6k", kind="sig", cloud="camera", n=6000, m=6000),
        dict(name="compi_6k", kind="compi", cloud="kinect", n=6000, m=6000),
        # nearest sources of every target under a pose, lists to the caller
        dict(name="knn8_200k", kind="knn", cloud="iso", n=200000, m=200000, k=8),
        # many registrations at once: coarse isotropic phase, then the
        # surface-covariance refinement on three resolutions
        dict(name="batch_64", kind="batch", cloud="trials", n=64, m=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("pose", "pose", "pose", "hess", "points", "cov_iteration", "sigma_iteration", "sig",
                       "compi", "knn", "loop", "batch"))
    if kind == "batch":
        return dict(kind=kind, cloud="trials", n=rng.randint(12, 64), m=0)
    if kind == "points":
        if rng.random() < 0.5:
            w = rng.randint(100, 320)
            return dict(kind=kind, cloud="views", n=w, m=rng.randint(w // 2, 3 * w // 4))
        return dict(kind=kind, cloud="contour", n=_log_int(rng, 300, 3000), m=_log_int(rng, 300, 3000))
    if kind == "pose":
        cloud = rng.choice(("contour", "iso", "camera"))
        lo, hi = {"contour": (300, 3000), "iso": (900, 200000), "camera": (900, 20000)}[cloud]
    elif kind in ("sig", "compi", "loop"):
        cloud = "kinect" if kind != "sig" else rng.choice(("kinect", "camera"))
        lo, hi = (460, 5400) if kind == "loop" else (460, 20000)
    else:
        cloud = "iso"
        lo, hi = {"hess": (900, 50000), "cov_iteration": (2000, 60000), "sigma_iteration": (2000, 200000),
                  "knn": (900, 200000)}[kind]
    n = _log_int(rng, lo, hi)
    # the two clouds of a registration are of similar size
    m = min(hi, max(lo, int(round(n * rng.uniform(0.6, 1.5)))))
    c = dict(kind=kind, cloud=cloud, n=n, m=m)
    if kind == "knn":
        c["k"] = rng.choice((1, 8, 8, 16, 32))
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _f32(a):
    return np.asarray(a, np.float64).astype(np.float32).astype(np.float64)


def _views(seed, w, h):
    """Two w x h depth views of one scene, 10 degrees apart at most."""
    rng = np.random.default_rng(seed)
    # the field of view of a 320-pixel image at f = 285
    P, C = W.depth_view(rng, W=w, H=h, f=285.0 * w / 320.0)
    R = W.random_rotation(rng, 10.0)
    t = rng.uniform(-0.05, 0.05, size=3)
    Q = P @ R.T + t
    CQ = np.einsum("ab,nbc,dc->nad", R, C, R)
    CQ = 0.5 * (CQ + np.transpose(CQ, (0, 2, 1)))
    return dict(X=Q.T.copy(), X_C=W.blocks(CQ), Y=P.T.copy(), Y_C=W.blocks(C), R_G=R, t_G=t)


def _clouds(case, seed):
    """The two clouds (FP32 values in FP64 arrays) and a pose a little off the
    true one, as in the middle of a registration."""
    n, m, cloud = case["n"], case["m"], case["cloud"]
    if cloud == "contour":
        d = W.config5_2d(seed, n, m)
    elif cloud == "iso":
        d = W.config3(seed, n, m)
    elif cloud == "camera":
        d = W.config2(seed, n, m)
    elif cloud == "kinect":
        d = W.kinect_like(seed, n, m)
    else:
        d = _views(seed, n, m)
    rng = np.random.default_rng([seed, 77])
    if cloud == "contour":
        R = W.rot2(math.radians(rng.uniform(1.0, 2.0))) @ d["R_G"]
        t = np.ravel(d["t_G"]) + rng.uniform(-0.003, 0.003, size=2)
    else:
        R = W.rot_axis_angle(rng.normal(size=3), math.radians(rng.uniform(1.0, 2.0))) @ d["R_G"]
        t = np.ravel(d["t_G"]) + rng.uniform(-0.003, 0.003, size=3)
    out = {k: _f32(d[k]) for k in ("X", "X_C", "Y", "Y_C")}
    out.update(R=R, t=t)
    return out


def _trials(case, seed):
    return [W.config4_trial(1000 * (seed % 1000000) + k, workers=1, covariances=True) for k in range(case["n"])]


class _Ctx:
    """A context that is freed with the state that holds it."""

    def __init__(self, d):
        _, self.h = dg.init(d["X"], d["X_C"], d["Y"], d["Y_C"])

    def __del__(self):
        try:
            dg.fr_m(self.h)
        except Exception:
            pass


class _Batch:
    def __init__(self, trials):
        self.b = dg.Batch(trials)

    def __del__(self):
        try:
            self.b.free()
        except Exception:
            pass


# the batched schedule of bench.py: sigma update and annealing on every 4th
# point, over-relaxed steps, then the refinement on three resolutions
_SCHEDULE = dict(max_iter=120, anneal=True, anneal_decay=0.95, sigma_update=True, tol_rot=1e-4, tol_trans=1e-4,
                 relax=1.9, coarse_iters=120, refine_iters=100, refine_coarse_iters=60, refine_mid_iters=20)


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, case=case)
    if kind == "batch":
        s["batch"] = _Batch(_trials(case, seed))
        return s
    d = _clouds(case, seed)
    s.update(R=d["R"], t=d["t"])
    if kind == "loop":
        # the whole loop starts from the caller's host arrays, 30 degrees off
        s.update(d, R=np.eye(3), t=np.zeros(3))
        return s
    s["ctx"] = _Ctx(d)
    if kind == "compi":
        s["sig"] = dg.update_sig(s["ctx"].h, s["R"], s["t"])
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind == "batch":
        return s["batch"].b.register(**_SCHEDULE)
    R, t = s["R"], s["t"]
    if kind == "loop":
        # the reference driver's settings
        return dg.DUGMA(s["X"], s["Y"], s["X_C"], s["Y_C"], R, t, Max_Iteration=300, accuracy_rotation=1e-4,
                        accuracy_translation=1e-8, accuracy_sig=1e-9)
    h = s["ctx"].h
    if kind == "pose":
        return dg.energy_grad(h, R, t)
    if kind == "hess":
        return dg.energy_grad_hess(h, R, t)
    if kind == "points":
        return dg.energy_grad_points(h, R, t)
    if kind == "cov_iteration":
        return dg.update_cov_knn(h, k=8), dg.energy_grad(h, R, t)
    if kind == "sigma_iteration":
        return dg.update_sigma_knn(h, k=8), dg.energy_grad(h, R, t)
    if kind == "sig":
        return dg.update_sig(h, R, t)
    if kind == "compi":
        return dg.compi(h, R, t, sig=s["sig"])
    return dg.knn(h, dg.KNN_TARGET_TO_SOURCE, s["case"]["k"], R, t)


def work(case):
    """Every point's record read once, every result written once; the
    arithmetic of every pair of the sum once (multiply-add 2, exp and rsq 1)."""
    kind, n, m = case["kind"], case["n"], case["m"]
    if kind == "batch":
        # trials of 500 to 8,000 points, mean product of the sizes about 7e6;
        # about 120 coarse passes (1/16 of the pairs, 25 operations a pair)
        # and the equivalent of 4 full ones of the refinement (107)
        return dict(bytes=n * 2700.0 * 2 * 64, flops=n * 7e6 * (120 / 16 * 25 + 4 * 107))
    D = 2 if case["cloud"] == "contour" else 3
    if case["cloud"] == "views":
        n = m = n * m
    pairs = float(n) * m
    full = case["cloud"] in ("camera", "views") or kind in ("cov_iteration", "points")
    rec = 4.0 * (D + (D * (D + 1) // 2 if full else 1))
    pair_flops = (107 if full else 36) if D == 3 else (45 if full else 25)
    read = rec * (n + m)
    if kind == "pose":
        return dict(bytes=read + 8 * 7, flops=pairs * pair_flops)
    if kind == "hess":
        return dict(bytes=read + 8 * 43, flops=pairs * (pair_flops + 20))
    if kind == "points":
        return dict(bytes=read + 8.0 * (D + D * D) * (n + m), flops=2 * pairs * pair_flops)
    if kind in ("cov_iteration", "sigma_iteration"):
        # positions in, covariances out, then the gradient's pass
        return dict(bytes=(12.0 + rec - 12.0 + 4.0) * (n + m) + read, flops=pairs * pair_flops)
    if kind == "sig":
        return dict(bytes=12.0 * (n + m) + 4, flops=pairs * 8)
    if kind == "compi":
        return dict(bytes=52.0 * (n + m) + 8 * 637, flops=pairs * 80)
    if kind == "loop":
        # about 60 iterations of both calls
        return dict(bytes=96.0 * (n + m), flops=60 * pairs * 88)
    return dict(bytes=12.0 * (n + m) + 8.0 * n * case["k"], flops=8.0 * (n + m) * case["k"])


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=_dev())


def _points(P, C):
    """(n, D) points and (n, D, D) covariances of the D x n, D x (D n) arrays."""
    return _t(P.T), _t(W.unblocks(C))


def _pair_sums(X, CX, Y, CY, want="pose"):
    """Sums over all pairs of e = det(S)^-1/2 exp(-d^T S^-1 d / 2) / (2 pi)^(D/2), d =
    x - y, S = CX + CY: for each x and each y [e (1), e w (D), e (w w^T - S^-1) (D, D)],
    w = S^-1 d.  Returns (A_x, A_y), each (count, 1 + D + D D)."""
    n, D = X.shape
    m = Y.shape[0]
    iso = bool((CX - CX[:, :1, :1] * torch.eye(D, dtype=CX.dtype, device=CX.device)).abs().max() == 0) and bool(
        (CY - CY[:, :1, :1] * torch.eye(D, dtype=CX.dtype, device=CX.device)).abs().max() == 0)
    norm = (2 * math.pi) ** (-D / 2)
    Ax = torch.zeros(n, 1 + D + D * D, dtype=torch.float64, device=X.device)
    Ay = torch.zeros(m, 1 + D + D * D, dtype=torch.float64, device=X.device)
    rows = max(1, int(1.5e8 // m))
    for i0 in range(0, n, rows):
        sl = slice(i0, min(n, i0 + rows))
        d = [X[sl, a, None] - Y[None, :, a] for a in range(D)]
        if iso:
            inv = 1.0 / (CX[sl, 0, 0, None] + CY[None, :, 0, 0])
            r2 = d[0] * d[0]
            for a in range(1, D):
                r2 = r2 + d[a] * d[a]
            e = norm * torch.exp(r2.mul_(inv).mul_(-0.5)) * (inv * torch.sqrt(inv) if D == 3 else inv)
            ew = e * inv
            w = d
            q = e.sum(1), e.sum(0)
            Ax[sl, 0] += q[0]
            Ay[:, 0] += q[1]
            for a in range(D):
                p = ew * w[a]
                Ax[sl, 1 + a] += p.sum(1)
                Ay[:, 1 + a] += p.sum(0)
            if want != "pose":
                sx, sy = ew.sum(1), ew.sum(0)
                ew2 = ew * inv
                for a in range(D):
                    for b in range(a, D):
                        p = ew2 * d[a] * d[b]
                        px, py = p.sum(1), p.sum(0)
                        if a == b:
                            px, py = px - sx, py - sy
                        for u, v in {(a, b), (b, a)}:
                            Ax[sl, 1 + D + D * u + v] += px
                            Ay[:, 1 + D + D * u + v] += py
            continue
        S = [[CX[sl, a, b, None] + CY[None, :, a, b] for b in range(D)] for a in range(D)]
        if D == 3:
            c = [[None] * 3 for _ in range(3)]
            for a in range(3):
                for b in range(a, 3):
                    r, s = [x for x in range(3) if x != a], [x for x in range(3) if x != b]
                    v = S[r[0]][s[0]] * S[r[1]][s[1]] - S[r[0]][s[1]] * S[r[1]][s[0]]
                    c[a][b] = c[b][a] = v if (a + b) % 2 == 0 else -v
            det = S[0][0] * c[0][0] + S[0][1] * c[0][1] + S[0][2] * c[0][2]
        else:
            c = [[S[1][1], -S[0][1]], [-S[0][1], S[0][0]]]
            det = S[0][0] * S[1][1] - S[0][1] * S[0][1]
        del S
        inv = 1.0 / det
        for a in range(D):
            for b in range(a, D):
                c[a][b] = c[b][a] = c[a][b] * inv
        w = []
        for a in range(D):
            v = c[a][0] * d[0]
            for b in range(1, D):
                v = v + c[a][b] * d[b]
            w.append(v)
        q = d[0] * w[0]
        for a in range(1, D):
            q = q + d[a] * w[a]
        e = norm * torch.sqrt(inv) * torch.exp(-0.5 * q)
        Ax[sl, 0] += e.sum(1)
        Ay[:, 0] += e.sum(0)
        for a in range(D):
            p = e * w[a]
            Ax[sl, 1 + a] += p.sum(1)
            Ay[:, 1 + a] += p.sum(0)
        for a in range(D):
            for b in range(a, D):
                p = e * (w[a] * w[b] - c[a][b])
                px, py = p.sum(1), p.sum(0)
                for u, v in {(a, b), (b, a)}:
                    Ax[sl, 1 + D + D * u + v] += px
                    Ay[:, 1 + D + D * u + v] += py
    return Ax, Ay


def _moved(d, CY=None):
    """Targets and transformed sources: (X, CX, R y + t, R CY R^T, R y)."""
    X, CX = _points(d["X"], d["X_C"])
    Y, C = _points(d["Y"], d["Y_C"])
    C = C if CY is None else CY
    R, t = _t(d["R"]), _t(d["t"])
    Ry = Y @ R.T
    return X, CX, Ry + t, torch.matmul(torch.matmul(R, C), R.T.contiguous()), Ry


def _pose_grad(Ay, z, S):
    """(E, gpose) from the sources' sums: z = R y, S = R CY R^T."""
    D = z.shape[1]
    g = Ay[:, 1:1 + D]  # dE/dx' = + sum e w (d = x - x')
    H = 0.5 * Ay[:, 1 + D:].reshape(-1, D, D)
    K = torch.matmul(H, S) - torch.matmul(S, H)
    if D == 3:
        rot = torch.linalg.cross(z, g)
        rot = rot + 2.0 * torch.stack([K[:, 2, 1], K[:, 0, 2], K[:, 1, 0]], dim=1)
        rot = rot.sum(0)
    else:
        rot = (g[:, 1] * z[:, 0] - g[:, 0] * z[:, 1] + 2.0 * K[:, 1, 0]).sum().reshape(1)
    return float(Ay[:, 0].sum()), torch.cat([rot, g.sum(0)]).cpu().numpy()


def _hessian(Ay, z):
    """Hessian of E in (w, t) for isotropic covariances."""
    g, B = Ay[:, 1:4], Ay[:, 4:].reshape(-1, 3, 3)
    # moving x' by u changes E by g.u + u^T B u / 2 (to second order)
    Z = torch.zeros(z.shape[0], 3, 3, dtype=torch.float64, device=z.device)
    Z[:, 0, 1], Z[:, 0, 2], Z[:, 1, 2] = z[:, 2], -z[:, 1], z[:, 0]
    Z = Z - torch.transpose(Z, 1, 2)  # w -> w x z = Z w
    J = torch.cat([Z, torch.eye(3, dtype=torch.float64, device=z.device).expand(z.shape[0], 3, 3)], dim=2)
    H = torch.matmul(torch.matmul(torch.transpose(J, 1, 2).contiguous(), B), J).sum(0)
    gz = g[:, :, None] * z[:, None, :]
    gz = gz.sum(0)
    H[:3, :3] += 0.5 * (gz + gz.T) - torch.trace(gz) * torch.eye(3, dtype=torch.float64, device=z.device)
    return H.cpu().numpy()


def _nearest(Q, P, k, skip_self):
    """(distances squared, indices) of the k nearest rows of P for each row of Q, nearest first."""
    dd, ii = [], []
    rows = max(1, int(2e8 // P.shape[0]))
    for i0 in range(0, Q.shape[0], rows):
        q = Q[i0:i0 + rows]
        d2 = (q[:, 0, None] - P[None, :, 0]) ** 2
        for a in range(1, Q.shape[1]):
            d2 += (q[:, a, None] - P[None, :, a]) ** 2
        if skip_self:
            r = torch.arange(q.shape[0], device=Q.device)
            d2[r, r + i0] = math.inf
        v, i = torch.topk(d2, k, dim=1, largest=False, sorted=True)
        dd.append(v)
        ii.append(i)
    return torch.cat(dd), torch.cat(ii)


def _iteration(d, surface):
    """Both clouds' covariances from their 8 nearest neighbours, then the gradient on them."""
    sig, cov = [], []
    for name in ("X", "Y"):
        P = _t(d[name].T)
        d2, idx = _nearest(P, P, 8, True)
        s = torch.sqrt(d2).mean(1)
        eye = torch.eye(3, dtype=torch.float64, device=P.device)
        if surface:
            c = P[idx] - P[idx].mean(1, keepdim=True)
            C = 0.5 * torch.matmul(torch.transpose(c, 1, 2).contiguous(), c) / 8 + (0.002 * s * s)[:, None, None] * eye
        else:
            C = (s * s)[:, None, None] * eye
        sig.append(s.cpu().numpy())
        cov.append(C)
    X, _, Yp, S, z = _moved(d, cov[1])
    _, Ay = _pair_sums(X, cov[0], Yp, S)
    return (sig[0], sig[1], None), _pose_grad(Ay, z, S)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("batch", "loop", "compi"):
        # whole registrations end where their own stopping rules say; compi's
        # 637 coefficients have no closed 64-bit form apart from the library's
        return None
    d = _clouds(case, seed)
    if kind in ("cov_iteration", "sigma_iteration"):
        return _iteration(d, kind == "cov_iteration")
    if kind == "knn":
        R, t = _t(d["R"]), _t(d["t"])
        d2, _ = _nearest(_t(d["X"].T), _t(d["Y"].T) @ R.T + t, case["k"], False)
        return None, d2.cpu().numpy()
    if kind == "sig":
        # mean over the targets of the nearest squared distance / 3, in
        # steps of 1e-6 (the definition's own quantisation)
        R, t = _t(d["R"]), _t(d["t"])
        d2, _ = _nearest(_t(d["X"].T), _t(d["Y"].T) @ R.T + t, 1, False)
        return float((torch.round(d2 / 3.0 * 1e6) / 1e6).mean())
    X, CX, Yp, S, z = _moved(d)
    if kind == "pose":
        _, Ay = _pair_sums(X, CX, Yp, S)
        return _pose_grad(Ay, z, S)
    if kind == "hess":
        _, Ay = _pair_sums(X, CX, Yp, S, want="all")
        E, g = _pose_grad(Ay, z, S)
        return E, g, _hessian(Ay, z)
    # per-point gradients
    Ax, Ay = _pair_sums(X, CX, Yp, S, want="all")
    D = z.shape[1]
    E, gpose = _pose_grad(Ay, z, S)
    R = _t(d["R"])
    g = Ay[:, 1:1 + D]
    H = 0.5 * Ay[:, 1 + D:].reshape(-1, D, D)
    G = (g[:, :, None] * z[:, None, :] + 2.0 * torch.matmul(H, S)).sum(0)
    gt = g.sum(0)
    if D == 3:
        gdT = torch.cat([gt, G.reshape(-1)])
    else:
        gdT = torch.cat([gt, (G[0, 0] + G[1, 1]).reshape(1), (G[1, 0] - G[0, 1]).reshape(1)])
    return dict(E=E, gpose=gpose, gX=(-Ax[:, 1:1 + D]).cpu().numpy(),
                gXC=(0.5 * Ax[:, 1 + D:].reshape(-1, D, D)).cpu().numpy(), gY=(g @ R).cpu().numpy(),
                gYC=torch.matmul(torch.matmul(R.T.contiguous(), H), R).cpu().numpy(), gdT=gdT.cpu().numpy())
