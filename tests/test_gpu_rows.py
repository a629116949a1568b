"""GPU tests of the entry points on sample-major rows (csrc/rows.hip): the
estimator's transform and predict against the feature-major entry points, bit
for bit."""
import numpy as np
import pytest
from numpy.testing import assert_array_equal

from tests.conftest import to_dev, to_np

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def q():
    return torch.cuda.current_stream()


def model_of(kd, centers):
    """A fitted model with the given centres."""
    k, d = centers.shape
    m = kd.KMeans(k, init=centers, n_init=1, max_iter=1)
    m.fit(np.concatenate([centers, centers]))
    m._centers_dev = to_dev(centers)
    return m


# edges of the 64-row waves and 256-row blocks, of the register buckets (8, 16,
# 32, 64, 128), of the 4-centre groups and 32-centre tiles; the last of each
# type is beyond the row kernel
@pytest.mark.parametrize("n,d,k,dt", [
    (1, 1, 1, np.float32), (63, 8, 4, np.float32), (65, 9, 5, np.float32),
    (256, 16, 31, np.float32), (257, 17, 33, np.float32), (1000, 32, 64, np.float32),
    (300, 33, 66, np.float32), (129, 64, 32, np.float32), (200, 65, 97, np.float32),
    (100, 128, 7, np.float32), (100, 129, 7, np.float32),
    (70, 7, 3, np.float64), (257, 16, 17, np.float64), (130, 33, 40, np.float64),
    (64, 64, 16, np.float64), (100, 65, 9, np.float64)])
def test_transform_equals_feature_major_distances(kd, torch_dev, n, d, k, dt):
    rng = np.random.default_rng(n + 3 * d + 5 * k)
    X = rng.standard_normal((n, d)).astype(dt)
    C = rng.standard_normal((k, d)).astype(dt)
    got = model_of(kd, C).transform(to_dev(X))
    D = torch.empty((k, n), dtype=got.dtype, device=torch_dev)
    kd.compute_centroid_to_sample_distances(to_dev(X.T), to_dev(C.T), D, 128, 32, q())[0].wait()
    assert got.shape == (n, k)
    assert_array_equal(to_np(got), to_np(D).T)
    exp = np.sqrt(((X[:, None, :].astype(np.float64) - C[None].astype(np.float64)) ** 2).sum(-1))
    # d squares and sums, a square root: at most d + 3 roundings of the value
    np.testing.assert_allclose(to_np(got), exp, rtol=(d + 3) * np.finfo(dt).eps)


# edges of the 32-row column blocks, of the feature buckets (4 to 64, then the
# tiled kernel's 80 to 128) and of the 32-centroid tiles; k = 2000 at d = 20 and
# k = 700 at d = 64 are beyond LDS, d = 129 beyond the row kernels
@pytest.mark.parametrize("n,d,k", [
    (1, 1, 1), (31, 3, 2), (33, 4, 33), (500, 5, 8), (511, 16, 32), (513, 17, 65),
    (1000, 32, 100), (700, 47, 200), (257, 48, 31), (300, 63, 40), (640, 64, 256),
    (300, 64, 700), (400, 20, 2000), (321, 65, 60), (200, 100, 96), (130, 128, 33),
    (90, 129, 12)])
def test_predict_equals_assignment(kd, torch_dev, n, d, k):
    rng = np.random.default_rng(7 * n + d + k)
    X = rng.standard_normal((n, d)).astype(np.float32)
    C = rng.standard_normal((k, d)).astype(np.float32)
    C[k // 2] = C[0]                  # an exact tie: the lower index wins
    got = model_of(kd, C).predict(to_dev(X))
    hn = torch.empty(k, device=torch_dev)
    lab = torch.empty(n, dtype=torch.int32, device=torch_dev)
    kd.half_l2_norm_squared(to_dev(C.T), hn, 128, q())
    kd.assignment(to_dev(X.T), to_dev(C.T), hn, lab, 8, 128, q())[0].wait()
    assert_array_equal(to_np(got), to_np(lab))


# several blocks of centres: one tile each, two each and a ragged last one
@pytest.mark.parametrize("n,d,k,dt", [(100, 5, 1000, np.float32), (25_600, 9, 200, np.float32),
                                      (30_001, 17, 201, np.float64), (65, 64, 17, np.float64)])
def test_transform_with_centres_over_blocks(kd, torch_dev, n, d, k, dt):
    rng = np.random.default_rng(n + k)
    X = rng.standard_normal((n, d)).astype(dt)
    C = rng.standard_normal((k, d)).astype(dt)
    got = model_of(kd, C).transform(to_dev(X))
    D = torch.empty((k, n), dtype=got.dtype, device=torch_dev)
    kd.compute_centroid_to_sample_distances(to_dev(X.T), to_dev(C.T), D, 128, 32, q())[0].wait()
    assert_array_equal(to_np(got), to_np(D).T)
