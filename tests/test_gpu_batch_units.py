"""How many waves share a unit of 64 targets depends on the number of units in
the batch and changes no result: copies of the same trials give the same bits at
every count (16, 8 and 4 waves a unit, and a wave per unit), with sizes at the
edges of 64-target units and 64-source blocks; one step agrees with the numpy
restatement."""
import numpy as np
import pytest

import dugma_amd as dg
from dugma_amd import workloads as W
from test_gpu_batch import numpy_step, small_trial

pytestmark = pytest.mark.gpu

# 271 units of the full clouds: 63 target pieces x 4 chunks for the first
SIZES = [(4000, 4000), (65, 129), (3, 64), (257, 63), (64, 65), (640, 1000)]
# units: 271 (16 waves each), 1,084 (8), 10,840 (4), 43,360 (a wave per unit; refinement 8 -> 4)
COPIES = (1, 4, 40, 160)


@pytest.fixture(scope="module")
def trials():
    out = []
    for q, (n, m) in enumerate(SIZES):
        tr = small_trial(90 + q, n, m, deg=8.0) if min(n, m) > 8 else None
        if tr is None:
            rng = np.random.default_rng(q)
            tr = dict(X=rng.normal(size=(3, n)), sX=np.full(n, 0.01), Y=rng.normal(size=(3, m)), sY=np.full(m, 0.02))
        rng = np.random.default_rng(500 + q)
        for p, s, c in (("X", "sX", "CX"), ("Y", "sY", "CY")):
            A = np.eye(3) + 0.4 * rng.normal(size=(tr[p].shape[1], 3, 3))
            tr[c] = tr[s][:, None, None] * (np.einsum("nab,ncb->nac", A, A) + 0.05 * np.eye(3))
        out.append(tr)
    return out


def _run(trials, copies, **kw):
    b = dg.Batch(trials * copies)
    try:
        return b.register(tol_rot=0.0, tol_trans=0.0, **kw)
    finally:
        b.free()


@pytest.mark.parametrize("kw", [dict(max_iter=3), dict(max_iter=3, sigma_update=False),
                                dict(max_iter=6, coarse_iters=4),
                                dict(max_iter=2, refine_iters=2, refine_coarse_iters=2, refine_mid_iters=1)],
                         ids=["sigma", "plain", "coarse", "refine"])
def test_units_shared_by_any_number_of_waves_give_the_same_bits(trials, kw):
    ref = _run(trials, COPIES[0], **kw)
    for copies in COPIES[1:]:
        got = _run(trials, copies, **kw)
        for key, v in ref.items():
            np.testing.assert_array_equal(got[key], np.concatenate([v] * copies), err_msg="%s x %d" % (key, copies))


@pytest.mark.parametrize("copies", COPIES)
def test_one_step_agrees_with_the_numpy_restatement(trials, copies):
    pick = [trials[0], trials[1], trials[3]]
    r = _run(pick, copies, max_iter=1, anneal=False, sigma_update=False)
    for k, tr in enumerate(pick):
        R, t = numpy_step(tr, np.eye(3), np.zeros(3))
        assert W.rotation_error_deg(r["R"][k], R) < 1e-4  # as test_one_step_matches_procrustes
        assert np.abs(r["t"][k] - t).max() < 1e-6
