"""The batched iteration's per-fit blocks at their edges: one centroid and one
feature, the largest tables, k that divides no stride, several empty clusters,
and more fits than a block has threads.  Every fit equals the single-fit
driver's bit for bit (labels, centroids, iterations)."""
import numpy as np
import pytest
from numpy.testing import assert_array_equal

from tests.test_gpu_batched import batched, single

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def problem(rng, n, d, k, empties):
    Xt = rng.standard_normal((d, n)).astype(np.float32)
    init = Xt[:, rng.choice(n, k, replace=False)].copy()
    far = rng.choice(k, min(empties, k - 1), replace=False)
    init[:, far] = 1e3
    return Xt, rng.uniform(0.5, 2.0, n).astype(np.float32), init, 0.0, 4


def same(probs):
    import kmeans_dpcpp_amd as kd
    got, _ = batched(kd, probs, 2)
    for p, g in zip(probs, got):
        exp = single(kd, *p)
        assert_array_equal(g[0], exp[0])
        assert_array_equal(g[1], exp[1])
        assert g[2] == exp[2]


@pytest.mark.parametrize("empties", [0, 1, 5])
def test_tables_at_their_edges(torch_dev, empties):
    rng = np.random.default_rng(empties)
    same([problem(rng, n, d, k, empties) for n, d, k in
          [(1, 1, 1), (1025, 1, 1), (2049, 64, 256), (5000, 63, 255), (3071, 33, 129),
           (1024, 1, 256), (4096, 17, 7), (300, 64, 1), (9001, 31, 200), (700, 3, 65)]])


def test_more_fits_than_a_block_has_threads(torch_dev):
    rng = np.random.default_rng(3)
    same([problem(rng, int(rng.integers(40, 900)), int(rng.integers(1, 20)),
                  int(rng.integers(1, 30)), i % 3) for i in range(300)])
