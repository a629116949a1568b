"""GPU tests of an iteration's end where its table takes several blocks: the
iteration that finds empty clusters, and those after the relocation, whose
shift sums all blocks have to reach before the loop decides to go on."""
import numpy as np
import pytest
from numpy.testing import assert_allclose

from oracle import lloyd_oracle as lo
from tests.conftest import to_dev, to_np

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def fit(kd, Xt, w, init, tol, max_iter, verbose):
    lab = torch.empty(Xt.shape[1], dtype=torch.int32, device="cuda")
    init_d = to_dev(init)
    res = torch.empty_like(init_d)
    n_iter, inertia = kd.kmeans_lloyd_driver(to_dev(Xt), to_dev(w), init_d, lab, res, tol, verbose,
                                             max_iter, 8, 128, 0.7, torch.cuda.current_stream())
    return to_np(lab), to_np(res), int(n_iter), float(inertia[0])


# tables of many tiles (d * padded k > 8192), the last beyond 1024 columns
@pytest.mark.parametrize("n,d,k", [(20_000, 96, 512), (8000, 300, 100), (12_000, 7, 1100)])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_relocation_in_a_table_of_many_tiles(kd, torch_dev, capfd, n, d, k, dt):
    """Empty clusters at both ends and in the middle of the table; sample j of
    blob j as the other centroids, so that no two of them share a blob.  The fit
    follows the oracle, and the verbose one (nothing enqueued ahead), to the
    roundings of sums of n values."""
    rng = np.random.default_rng(n + d)
    centers = rng.uniform(-10, 10, (k, d))
    blob = np.concatenate([np.arange(k), rng.integers(0, k, n - k)])
    Xt = np.ascontiguousarray((centers[blob] + 0.3 * rng.standard_normal((n, d))).T.astype(dt))
    w = rng.uniform(0.5, 2, n).astype(dt)
    init = Xt[:, :k].copy()
    for j, c in enumerate((0, 1, k // 2, k - 2, k - 1)):
        init[:, c] = 1e4 * (j + 1)
    for max_iter in (1, 6):
        lab, C, it, inertia = fit(kd, Xt, w, init, 0.0, max_iter, False)
        elab, eC, eit, einertia = lo.kmeans_lloyd(Xt, w, init, 0.0, max_iter, dtype=np.float64)
        slab, sC, sit, sinertia = fit(kd, Xt, w, init, 0.0, max_iter, True)
        capfd.readouterr()
        eps = np.finfo(dt).eps
        # a mean of values up to |x|: quantised or rounded products and sums
        tol = 32 * eps * np.abs(Xt).max()
        assert it == sit
        assert np.abs(C - sC).max() <= tol
        assert np.array_equal(lab, slab)
        # (with tol = 0, FP32 sums in another order end a fit at another iteration;
        # the centroids are the fixed point then)
        assert it == eit if max_iter == 1 else it >= 1
        assert np.abs(C - eC).max() <= tol
        assert np.array_equal(lab, elab)
        assert_allclose(inertia, einertia, rtol=64 * eps * d)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_fits_after_a_relocation_keep_their_iterations(kd, torch_dev, dt):
    """A loop of many iterations after the relocation: the same number of them,
    the same centroids, time after time, with another stream at work."""
    n, d, k = 30_000, 40, 300
    Xt, init = lo.gaussian_blobs(n, d, k, seed=5, std=3.0, dtype=dt)
    init = init.copy()
    init[:, [0, 17, 150, 298, 299]] = 1e4
    w = np.ones(n, dt)
    other = torch.cuda.Stream()
    a = torch.randn(2048, 2048, device="cuda")
    got = []
    for _ in range(6):
        with torch.cuda.stream(other):
            for _ in range(20):
                torch.mm(a, a)
        got.append(fit(kd, Xt, w, init, 1e-4, 40, False))
    torch.cuda.synchronize()
    for g in got[1:]:
        assert g[2] == got[0][2]
        assert_allclose(g[1], got[0][1], rtol=0, atol=64 * np.finfo(dt).eps * np.abs(Xt).max())
