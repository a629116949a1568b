"""GPU tests of the float32 kernels for more than 128 features or more than
32768 clusters (csrc/lloyd_wide.hip): labels against the C restatement, whose
sequential FMA chain they follow bit for bit, and fits against an FP64 update."""
import numpy as np
import pytest
from numpy.testing import assert_array_equal

from oracle import c_oracle as co
from oracle import lloyd_oracle as lo
from tests.conftest import check_label_mismatches, fp64_update, to_dev, to_np

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def q():
    return torch.cuda.current_stream()


# edges of the 32-sample columns and 128-sample blocks, of the 16-feature
# chunks, of the 32-centroid tiles and of one launch's 8 tiles
SHAPES = [(1, 129, 1), (31, 144, 32), (33, 145, 33), (127, 160, 65), (129, 303, 100),
          (1000, 300, 256), (257, 131, 257), (640, 1025, 520), (300, 2, 32801),
          (524_300, 130, 40)]     # the last: two column blocks per wave


@pytest.mark.parametrize("n,d,k", SHAPES)
@pytest.mark.parametrize("it", [torch.int32, torch.int64])
def test_labels_equal_the_sequential_chain(kd, torch_dev, n, d, k, it):
    rng = np.random.default_rng(n * 7 + d + k)
    Xt = rng.standard_normal((d, n)).astype(np.float32)
    C = rng.standard_normal((d, k)).astype(np.float32)
    C[:, k // 2] = C[:, 0]            # an exact tie: the lower index wins
    hn = co.half_norm(C)
    lab = torch.full((n,), -1, dtype=it, device=torch_dev)
    kd.assignment(to_dev(Xt), to_dev(C), to_dev(hn), lab, 8, 128, q())[0].wait()
    assert_array_equal(to_np(lab), co.assign(Xt, C, hn))


def test_labels_pass_over_nan(kd, torch_dev):
    rng = np.random.default_rng(3)
    n, d, k = 200, 150, 40
    Xt = rng.standard_normal((d, n)).astype(np.float32)
    Xt[7, 5] = np.nan                 # every score NaN: label 0
    Xt[149, 6] = np.inf
    C = rng.standard_normal((d, k)).astype(np.float32)
    C[0, 0] = np.nan                  # a centroid that never wins
    hn = co.half_norm(C)
    lab = torch.full((n,), -1, dtype=torch.int32, device=torch_dev)
    kd.assignment(to_dev(Xt), to_dev(C), to_dev(hn), lab, 8, 128, q())[0].wait()
    assert_array_equal(to_np(lab), co.assign(Xt, C, hn))


@pytest.mark.parametrize("n,d,k", [(5000, 129, 1), (4097, 300, 100), (3001, 520, 33),
                                   (2500, 140, 2048)])
def test_driver_update(kd, torch_dev, n, d, k):
    """One iteration from given centroids: the labels of the sequential chain
    and the FP64 update of those labels, within the float32 roundings of each
    product w x, of the blocks' totals and their sums over blocks and copies,
    of the count and of the quotient."""
    rng = np.random.default_rng(d + k)
    Xt = rng.standard_normal((d, n)).astype(np.float32)
    init = Xt[:, :k].copy()
    w = rng.uniform(0.5, 2.0, n).astype(np.float32)
    lab0 = co.assign(Xt, init, co.half_norm(init))
    res = torch.empty((d, k), device=torch_dev)
    lab = torch.empty(n, dtype=torch.int32, device=torch_dev)
    it, _ = kd.kmeans_lloyd_driver(to_dev(Xt), to_dev(w), to_dev(init), lab, res, 0.0, False,
                                   1, 8, 128, 0.7, q())
    assert it == 1
    exp, cnt = fp64_update(Xt, w, lab0, k)
    got = to_np(res)
    # |error of a sum| <= (one product rounding + at most 8 partial sums) x
    # 2^-24 of the cluster's sum of |w x|; likewise the count and the quotient
    mag = np.stack([np.bincount(lab0, np.abs(Xt[f]).astype(np.float64) * w, minlength=k)
                    for f in range(d)])
    assert np.all(np.abs(got - exp) <= 20 * 2.0 ** -24 * mag / cnt)
    assert_array_equal(to_np(lab), co.assign(Xt, got, co.half_norm(got)))


def test_fused_step_follows_its_labels(kd, torch_dev):
    """The single-step entry point at d > 128: the assignment's labels, exact
    unit-weight counts, sums added to what the copies held."""
    n, d, k, copies = 6000, 200, 70, 3
    Xt, init = lo.gaussian_blobs(n, d, k, seed=4, dtype=np.float32)
    hn = co.half_norm(init)
    ids = torch.empty(n, dtype=torch.int32, device=torch_dev)
    cp = torch.full((copies, d, k), 0.5, device=torch_dev)
    scp = torch.full((copies, k), 2.0, device=torch_dev)
    kd.fused_lloyd_single_step(to_dev(Xt), torch.ones(n, device=torch_dev), to_dev(init),
                               to_dev(hn), ids, cp, scp, 8, 256, q())[0].wait()
    lab = to_np(ids)
    assert_array_equal(lab, co.assign(Xt, init, hn))
    assert_array_equal(to_np(scp).sum(axis=0) - 2.0 * copies, np.bincount(lab, minlength=k))
    sums = to_np(cp).astype(np.float64).sum(axis=0) - 0.5 * copies
    exp = np.stack([np.bincount(lab, Xt[f].astype(np.float64), minlength=k) for f in range(d)])
    assert np.abs(sums - exp).max() <= 1e-5 * np.abs(exp).max()


# both sides of the rule between the two updates from labels: k = 1024, n = 8 k,
# and the largest k of which two rows of sums fit LDS (9726)
@pytest.mark.parametrize("n,d,k", [(2050, 96, 1024), (2050, 96, 1025), (8200, 96, 1025),
                                   (77_807, 5, 9726), (77_808, 5, 9726), (77_816, 5, 9727)])
def test_both_updates_of_the_fused_step(kd, torch_dev, n, d, k):
    rng = np.random.default_rng(n + k)
    Xt = rng.standard_normal((d, n)).astype(np.float32)
    init = np.ascontiguousarray(Xt[:, :k])
    w = rng.uniform(0.5, 2.0, n).astype(np.float32)
    hn = co.half_norm(init)
    ids = torch.empty(n, dtype=torch.int32, device=torch_dev)
    cp = torch.zeros((2, d, k), device=torch_dev)
    scp = torch.zeros((2, k), device=torch_dev)
    kd.fused_lloyd_single_step(to_dev(Xt), to_dev(w), to_dev(init), to_dev(hn), ids, cp, scp,
                               8, 256, q())[0].wait()
    lab = to_np(ids)
    # (the tiled kernel's chain starts from the half norm)
    check_label_mismatches(Xt, init, lab, co.assign(Xt, init, hn), 4)
    cnt = np.bincount(lab, w, minlength=k)
    # m values a cluster: each product and each addition rounds once
    m = np.bincount(lab, minlength=k)
    got = to_np(scp).astype(np.float64).sum(axis=0)
    assert np.all(np.abs(got - cnt) <= (m + 4) * 2.0 ** -24 * cnt)
    sums = to_np(cp).astype(np.float64).sum(axis=0)
    for f in range(d):
        v = Xt[f].astype(np.float64) * w
        exp, mag = (np.bincount(lab, a, minlength=k) for a in (v, np.abs(v)))
        assert np.all(np.abs(sums[f] - exp) <= (m + 4) * 2.0 ** -24 * mag)


# few clusters (copies of the sums by lane), few samples (more groups of rows),
# rows that are no whole step of eight, one sample
@pytest.mark.parametrize("n,d,k", [(1, 131, 1), (65, 130, 2), (700, 513, 3), (3000, 800, 8),
                                   (2049, 136, 31), (10_000, 129, 33), (4097, 305, 63),
                                   (5000, 143, 64), (40_000, 128, 2), (2048, 97, 5)])
@pytest.mark.parametrize("kind", ["plain", "spread", "zero start", "small weights"])
def test_sums_of_few_clusters(kd, torch_dev, n, d, k, kind):
    """The fused step's sums against FP64 ones of its labels, also where values lie
    outside the window that the first samples of a block set (spread), where those
    have no weight, and where the weights are far from 1."""
    rng = np.random.default_rng(n + d + k)
    Xt = rng.standard_normal((d, n)).astype(np.float32)
    w = rng.uniform(0.5, 2.0, n).astype(np.float32)
    if kind == "spread":
        Xt *= (10.0 ** rng.uniform(-15, 9, n)).astype(np.float32)
    elif kind == "zero start":
        w[:64] = 0.0
    elif kind == "small weights":
        w *= np.float32(1e-9)
    # coordinates far below the samples', as of centred data
    init = (1e-3 * rng.standard_normal((d, k))).astype(np.float32)
    hn = co.half_norm(init)
    ids = torch.empty(n, dtype=torch.int32, device=torch_dev)
    cp = torch.zeros((2, d, k), device=torch_dev)
    scp = torch.zeros((2, k), device=torch_dev)
    kd.fused_lloyd_single_step(to_dev(Xt), to_dev(w), to_dev(init), to_dev(hn), ids, cp, scp,
                               8, 256, q())[0].wait()
    lab = to_np(ids)
    m = np.bincount(lab, minlength=k)
    # m values a cluster, each rounded in its product, at most each in its addition
    cnt = np.bincount(lab, w, minlength=k)
    assert np.all(np.abs(to_np(scp).astype(np.float64).sum(axis=0) - cnt)
                  <= (m + 4) * 2.0 ** -24 * cnt)
    sums = to_np(cp).astype(np.float64).sum(axis=0)
    for f in range(d):
        v = Xt[f].astype(np.float64) * w
        exp, mag = (np.bincount(lab, a, minlength=k) for a in (v, np.abs(v)))
        assert np.all(np.abs(sums[f] - exp) <= (m + 4) * 2.0 ** -24 * mag + 1e-40)
