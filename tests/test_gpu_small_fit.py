"""GPU tests of the one-block fit (small_loop_krn): every output equals, bit for
bit, that of the kernels of one iteration each, which KMD_NO_SMALLK=1 selects."""
import numpy as np
import pytest
from numpy.testing import assert_array_equal

from tests.conftest import to_dev, to_np

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def fit(kd, Xt, w, init, tol, max_iter, it=torch.int32):
    init_d = to_dev(init)
    res = torch.empty_like(init_d)
    lab = torch.full((Xt.shape[1],), -1, dtype=it, device="cuda")
    n_iter, inertia = kd.kmeans_lloyd_driver(to_dev(Xt), to_dev(w), init_d, lab, res, tol, False,
                                             max_iter, 8, 128, 0.7,
                                             torch.cuda.current_stream())
    return to_np(lab), to_np(res), int(n_iter), float(inertia[0])


def both(kd, monkeypatch, *args, **kw):
    got = fit(kd, *args, **kw)
    monkeypatch.setenv("KMD_NO_SMALLK", "1")
    exp = fit(kd, *args, **kw)
    monkeypatch.delenv("KMD_NO_SMALLK")
    for g, e in zip(got, exp):
        assert_array_equal(g, e)
    return got


def blobs(n, d, k, seed):
    rng = np.random.default_rng(seed)
    c = rng.uniform(-5, 5, (k, d))
    X = c[rng.integers(0, k, n)] + rng.standard_normal((n, d))
    return np.ascontiguousarray(X.T.astype(np.float32)), rng.uniform(0.5, 2, n).astype(np.float32)


# edges of the 64-sample waves and 1024-sample slots, of the feature buckets (8,
# 16, 32, 64) and centroid groups (4, 8, 16, 32), of the two sum blocks (4096);
# the last two are beyond the kernel's rule
@pytest.mark.parametrize("n,d,k", [
    (1, 1, 1), (63, 3, 2), (65, 8, 4), (1000, 16, 8), (1024, 9, 5), (1025, 16, 9),
    (1000, 32, 32), (777, 33, 4), (1024, 64, 16), (2000, 16, 32), (4096, 8, 17),
    (4097, 5, 3), (8192, 8, 4), (8193, 8, 4), (4000, 8, 32)])
@pytest.mark.parametrize("it", [torch.int32, torch.int64])
def test_small_fit_equals_separate_kernels(kd, torch_dev, monkeypatch, n, d, k, it):
    Xt, w = blobs(n, d, k, n + d + k)
    got = both(kd, monkeypatch, Xt, w, Xt[:, :k].copy(), 1e-5, 60, it=it)
    assert got[2] >= 1
    for max_iter in (0, 1, 2):
        both(kd, monkeypatch, Xt, w, Xt[:, :k].copy(), 0.0, max_iter, it=it)


@pytest.mark.parametrize("max_iter", [1, 2, 30])
def test_small_fit_relocates(kd, torch_dev, monkeypatch, max_iter):
    """Far initial centroids leave clusters empty in the first iteration."""
    Xt, w = blobs(900, 7, 6, 3)
    init = Xt[:, :6].copy()
    init[:, 1] = 1e3
    init[:, 4] = -1e3
    got = both(kd, monkeypatch, Xt, w, init, 1e-6, max_iter)
    if max_iter == 30:
        assert len(np.unique(got[0])) == 6


@pytest.mark.parametrize("bad", ["inf", "range", "weights"])
def test_small_fit_hands_over_what_fixed_point_cannot_hold(kd, torch_dev, monkeypatch, bad):
    Xt, w = blobs(500, 6, 3, 9)
    if bad == "inf":
        Xt[2, 7] = np.inf
        w[7] = 0.0
    elif bad == "range":
        Xt[1] *= 1e-4
        Xt[1, 5] = 1e6
    else:
        w[3] = 1e-6
    init = Xt[:, 20:23].copy()
    got = fit(kd, Xt, w, init, 1e-5, 20)
    monkeypatch.setenv("KMD_NO_SMALLK", "1")
    exp = fit(kd, Xt, w, init, 1e-5, 20)
    monkeypatch.delenv("KMD_NO_SMALLK")
    # FP32 sums, whose order is not fixed: 500 additions of one rounding each
    assert_array_equal(got[0], exp[0])
    np.testing.assert_allclose(got[1], exp[1], rtol=500 * 2.0 ** -24, atol=1e-3)


def test_small_fit_has_no_step_to_time_and_no_plan(kd, torch_dev):
    """One launch is the whole fit, so there is no fused step to report; plans
    are timed with separate launches and kept for the sizes that have them."""
    n, d, k = 1500, 10, 6
    Xt, w = blobs(n, d, k, 11)
    Xd, wd, init = to_dev(Xt), to_dev(w), to_dev(Xt[:, :k].copy())

    def stats(Xd, wd):
        lab = torch.empty(Xd.shape[1], dtype=torch.int32, device="cuda")
        it, _, st = kd.kmeans_lloyd_driver_ex(Xd, wd, init.clone(), lab, torch.empty_like(init),
                                              0.0, False, 5, "fp32", torch.cuda.current_stream())
        return int(it), st

    it, st = stats(Xd, wd)
    assert it >= 1 and st["path"] == "fp32-mfma"
    assert st["fused_launches"] == 0 and st["fused_kernel_ms"] == 0.0
    tuned = kd.autotune(Xd, wd, init, "fp32", 2, torch.cuda.current_stream())
    assert all(c[3] > 0 for c in tuned["candidates"])
    it, st = stats(Xd, wd)
    assert st["fused_launches"] == 0
    # 9000 samples are beyond the rule: a launch an iteration
    Xt, w = blobs(9000, d, k, 11)
    it, st = stats(to_dev(Xt), to_dev(w))
    assert st["fused_launches"] == it and st["fused_kernel_ms"] > 0
