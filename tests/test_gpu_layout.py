"""Sample-major copies and BF16 operands of the tiled path at the edges of
their blocks, and the inertia with centroids staged by pieces."""
import numpy as np
import pytest
from numpy.testing import assert_array_equal

from tests.conftest import check_label_mismatches, to_dev, to_np

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def fit(kd, Xt, w, init, precision):
    lab = torch.zeros(Xt.shape[1], dtype=torch.int32, device="cuda")
    res = torch.zeros_like(init)
    stats = kd.kmeans_lloyd_driver_ex(Xt, w, init.clone(), lab, res, 0.0, False, 1, precision,
                                      torch.cuda.current_stream())[2]
    assert stats["path"] == {"fp32": "tiled-fp32", "bf16": "tiled-bf16+rescore"}[precision]
    return to_np(lab), to_np(res)


@pytest.mark.parametrize("n,d", [(33000, 33), (33001, 65), (33023, 100), (32833, 128),
                                 (33063, 127)])
def test_copies_of_the_samples(kd, torch_dev, n, d):
    """One iteration: centroids are the means of the FP64 sums over X_r, and the
    BF16 labels (bound from xnb, candidates from xb) are the FP32 ones."""
    g = np.random.default_rng(n)
    k = 600
    X = g.standard_normal((d, n)).astype(np.float32)
    Xt, w = to_dev(X), torch.ones(n, device=torch_dev)
    init = Xt[:, :k].contiguous()
    lab, C = fit(kd, Xt, w, init, "fp32")
    lab16, C16 = fit(kd, Xt, w, init, "bf16")
    check_label_mismatches(X, to_np(init), lab16, lab, 4)
    # rounding of one mean to FP32, and fixed-point sums within 2^-20 of the
    # largest value a sample
    first = ((0.5 * (to_np(init).astype(np.float64) ** 2).sum(0))[:, None]
             - to_np(init).astype(np.float64).T @ X.astype(np.float64)).argmin(0)
    cnt = np.bincount(first, minlength=k)
    sums = np.stack([np.bincount(first, X[f].astype(np.float64), minlength=k) for f in range(d)])
    ok = cnt > 0
    exp = sums[:, ok] / cnt[ok]
    for got in (C, C16):
        bad = np.abs(got[:, ok] - exp) > 2.0 ** -20 * np.abs(X).max()
        # a sample on a tie of the first assignment may be in either cluster
        assert bad.any(axis=0).sum() <= 4


@pytest.mark.parametrize("n,d,k", [(524288, 9, 2048), (524287, 9, 2048), (524545, 17, 2049),
                                   (77001, 64, 300), (600000, 33, 600), (530001, 8, 2000),
                                   (1048577, 4, 4096)])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("it", [np.int32, np.int64])
def test_inertia_by_pieces(kd, torch_dev, n, d, k, dt, it):
    """Bit for bit what the samples give in small parts, whose centroids are
    gathered from memory; a label out of range gives NaN."""
    g = np.random.default_rng(n + k)
    X = to_dev(g.standard_normal((d, n)).astype(dt))
    C = to_dev(g.standard_normal((d, k)).astype(dt))
    w = to_dev(g.uniform(0.5, 2, n).astype(dt))
    ids = g.integers(0, k, n).astype(it)
    ids[5], ids[n - 2] = -1, k
    ids = to_dev(ids)

    def run(X, w, ids):
        out = torch.empty(ids.shape[0], dtype=X.dtype, device=torch_dev)
        kd.compute_inertia(X, w, C, ids, out, work_group_size=256,
                           sycl_queue=torch.cuda.current_stream())[0].wait()
        return to_np(out)

    whole = run(X, w, ids)
    assert np.isnan(whole[[5, n - 2]]).all() and np.isfinite(whole).sum() == n - 2
    for a in (0, 3 * n // 7, n - 1000):
        b = min(n, a + 1000)
        assert_array_equal(whole[a:b], run(X[:, a:b].contiguous(), w[a:b].contiguous(),
                                           ids[a:b].contiguous()))
