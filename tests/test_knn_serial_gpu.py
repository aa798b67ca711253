"""The sequential kernel that overflowing queries and k > 64 go to, at the edges of its chunks (256
rows), wavefronts and row widths, against the oracle: rows that each enter the heap, equal rows,
non-finite values; indices in heap order and distance bits."""
import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu

METRICS = [(S.SC_EUCLIDIAN, O.EUCLIDIAN), (S.SC_MANHATTAN, O.MANHATTAN), (S.SC_MINKOWSKI, O.MINKOWSKI)]


def check(x, y, k, metric, om, mode=S.SC_PLAIN_FP64):
    gi, gd, gc = S.Index(x).knn(y, k, metric, 3, mode)
    over = S.last_stats()["overflow_queries"]
    oi, od, oc = O.linear_find_batch(x, y, k, om, 3)
    np.testing.assert_array_equal(gc, oc)
    for r in range(len(y)):
        c = int(oc[r])
        np.testing.assert_array_equal(gi[r, :c], oi[r, :c])
        if om == O.MINKOWSKI:  # pow differs in its last bits between host and device
            np.testing.assert_allclose(gd[r, :c], od[r, :c], rtol=1e-13)
        else:
            np.testing.assert_array_equal(gd[r, :c].view(np.uint64), od[r, :c].view(np.uint64))
    return over


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("metric,om", METRICS)
@pytest.mark.parametrize("n,d,k", [(65, 1, 65), (255, 5, 70), (257, 2, 90), (511, 3, 100), (512, 16, 512), (513, 17, 66), (1_025, 40, 200),
                                   (1_600, 33, 70), (700, 4_100, 90), (700, 8_200, 90)])
def test_large_k(n, d, k, metric, om, dtype):
    rng = np.random.default_rng(n + d)
    x, y = rng.normal(size=(n, d)).astype(dtype), rng.normal(size=(3, d)).astype(dtype)
    if n > 100:
        x[3::40, 0], x[5::50, d - 1], y[1, 0] = np.nan, np.inf, np.nan
    assert check(x, y, k, metric, om) == 3


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", ["approaching", "equal", "few values"])
@pytest.mark.parametrize("n,q,d,k", [(70_001, 2, 5, 1), (66_000, 33, 16, 20), (70_100, 7, 40, 64)])
def test_overflowing_queries(n, q, d, k, case, dtype):
    rng = np.random.default_rng(n)
    y = 0.01 * rng.normal(size=(q, d))
    if case == "approaching":  # every row enters
        x = np.linspace(50.0, 1.0, n)[:, None] * np.ones((1, d))
    elif case == "equal":
        x = np.ones((n, d))
    else:
        x, y = rng.integers(0, 2, size=(n, d)).astype(float), rng.integers(0, 2, size=(q, d)).astype(float)
    x, y = x.astype(dtype), y.astype(dtype)
    over = check(x, y, k, S.SC_EUCLIDIAN, O.EUCLIDIAN)
    if case != "few values":
        assert over == q
    if dtype == np.float32:
        check(x, y, k, S.SC_MANHATTAN, O.MANHATTAN, S.SC_MIXED)
        if k <= 32:
            check(x, y, k, S.SC_EUCLIDIAN, O.EUCLIDIAN, S.SC_MIXED)
