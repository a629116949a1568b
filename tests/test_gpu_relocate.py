"""Order of the far samples in the relocation of empty clusters: one block's
selection (n <= 262144, m <= 512) and the general one beyond, against the
oracle.  The samples' rows are set to small whole numbers, so that the moved
sums are exact and every result is compared bit by bit."""
import numpy as np
import pytest
from numpy.testing import assert_array_equal

from oracle import lloyd_oracle as lo
from tests.conftest import to_dev, to_np

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,m,kind", [
    (1, 1, "random"), (3, 3, "random"), (512, 512, "random"), (1023, 511, "random"),
    (1025, 512, "ties"), (1025, 513, "ties"), (2048, 5, "equal"), (2049, 5, "equal"),
    (5000, 400, "equal"), (9001, 64, "ties"), (9001, 512, "zeros"), (5000, 3, "inf"), (50000, 512, "ties"),
    (262144, 512, "random"), (262145, 40, "ties")])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_far_order(kd, torch_dev, n, m, kind, dt):
    rng = np.random.default_rng(n + m)
    d, k = 3, m + 5
    Xt = rng.integers(-8, 9, size=(d, n)).astype(dt)
    w = rng.integers(1, 4, size=n).astype(dt)
    lab = rng.integers(0, 5, size=n)
    if kind == "random":
        sq = rng.random(n)
    elif kind == "ties":
        sq = rng.integers(0, 50, size=n) / 8.0
    elif kind == "equal":
        sq = np.full(n, 0.5)
    elif kind == "zeros":
        sq = np.zeros(n)
        sq[rng.choice(n, m // 2, replace=False)] = rng.random(m // 2)
    else:
        sq = rng.random(n)
        sq[rng.choice(n, 4, replace=False)] = np.inf
    sq = sq.astype(dt)
    sums = rng.integers(-100, 100, size=(d, k)).astype(dt)
    sizes = np.full(k, 4.0 * n).astype(dt)
    lst = np.zeros(k, dtype=np.int64)
    lst[:m] = np.arange(5, k)
    Ce, se, ie = lo.relocate_empty_clusters(m, Xt, w, lab, lst, sq, sums, sizes, sq)
    Cd, sd, idd = to_dev(sums), to_dev(sizes), to_dev(sq)
    kd.relocate_empty_clusters(m, to_dev(Xt), to_dev(w), to_dev(lab), to_dev(lst), to_dev(sq),
                               Cd, sd, idd, 256, torch.cuda.current_stream())[0].wait()
    assert_array_equal(to_np(Cd), Ce)
    assert_array_equal(to_np(sd), se)
    assert_array_equal(to_np(idd), ie)


# NaN distances: some beside enough others, fewer others than m, none; on both
# sides of the one-block rule (n = 262144, m = 512), and with the others in the
# samples of few threads, whose list overflows
@pytest.mark.parametrize("n,m,others", [
    (50, 3, 40), (50, 3, 2), (50, 1, 0), (50, 4, 0), (3000, 512, 600), (3000, 512, 300),
    (3000, 513, 600), (3000, 513, 300), (9001, 5, 4), (262144, 40, 262100),
    (262144, 40, 13), (262145, 40, 262100), (262145, 40, 13), (262145, 40, 0),
    (262145, 1, 7), (262144, 300, "few threads")])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_nan_is_never_far(kd, torch_dev, n, m, others, dt):
    rng = np.random.default_rng(n + m)
    d, k = 3, m + 5
    Xt = rng.integers(-8, 9, size=(d, n)).astype(dt)
    w = rng.integers(1, 4, size=n).astype(dt)
    lab = rng.integers(0, 5, size=n)
    sq = np.full(n, np.nan, dtype=dt)
    if others == "few threads":
        at = np.flatnonzero(np.arange(n) % 1024 < 20)
    else:
        at = rng.choice(n, others, replace=False)
    sq[at] = rng.random(at.size)
    if at.size > 3:
        sq[at[:2]] = 0.5
        sq[at[2]] = np.inf
    sq[::3] = np.where(np.isnan(sq[::3]), -sq[::3], sq[::3])      # NaN of both signs
    sums = rng.integers(-100, 100, size=(d, k)).astype(dt)
    sizes = np.full(k, 4.0 * n).astype(dt)
    lst = np.zeros(k, dtype=np.int64)
    lst[:m] = np.arange(5, k)
    # the oracle's order has NaN last: as many as there are other distances
    Ce, se, ie = lo.relocate_empty_clusters(min(m, at.size), Xt, w, lab, lst, sq, sums, sizes, sq)
    Cd, sd, idd = to_dev(sums), to_dev(sizes), to_dev(sq)
    kd.relocate_empty_clusters(m, to_dev(Xt), to_dev(w), to_dev(lab), to_dev(lst), to_dev(sq),
                               Cd, sd, idd, 256, torch.cuda.current_stream())[0].wait()
    assert_array_equal(to_np(Cd), Ce)
    assert_array_equal(to_np(sd), se)
    assert_array_equal(to_np(idd), ie)
