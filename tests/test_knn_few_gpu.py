"""Few queries over few rows: the two-launch form against the general one (the same queries among
more than 1,024) and, for the reference's own order, the oracle; bit for bit."""
import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S
from test_knn_f64_gpu import _data as matrix_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metric", [S.SC_EUCLIDIAN, S.SC_MANHATTAN])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,q,d,k", [(1, 1, 1, 1), (5, 2, 3, 5), (63, 1, 16, 7), (64, 3, 17, 64), (255, 1, 8, 2),
                                     (257, 5, 33, 20), (1023, 1, 4, 64), (1024, 2, 5, 1), (1025, 4, 40, 10),
                                     (5000, 7, 100, 3), (65536, 1, 2, 33)])
def test_few_equals_general(n, q, d, k, dtype, metric):
    rng = np.random.default_rng(n + d)
    x, y = rng.normal(size=(n, d)), rng.normal(size=(q, d))
    x = np.rint(4 * x) / 4 if d < 6 else x  # narrow rows: many equal distances
    if n > 200:
        x[3::17, 0], x[5::41, d - 1] = np.nan, np.inf
        x[7::53] *= 1e200 if dtype == np.float64 else 1e25
    if q > 3:
        y[1, 0], y[2] = np.nan, y[2] * (1e200 if dtype == np.float64 else 1e25)
    with np.errstate(over="ignore"):
        x, y = x.astype(dtype), y.astype(dtype)
    ix = S.Index(x)
    few = ix.knn(y, k, metric)
    many = ix.knn(np.tile(y, (1024 // q + 1, 1)), k, metric)
    for a, b in zip(few, many):
        np.testing.assert_array_equal(np.asarray(a).view(np.uint8), np.ascontiguousarray(b[:q]).view(np.uint8))
    oi, od = O.linear_find(x, y[0], k, O.EUCLIDIAN if metric == S.SC_EUCLIDIAN else O.MANHATTAN)
    c = int(few[2][0])
    np.testing.assert_array_equal(few[0][0][:c], oi)
    np.testing.assert_array_equal(few[1][0][:c].view(np.uint64), np.asarray(od).view(np.uint64))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", ["sorted by class", "approaching", "ties", "far from the origin",
                                  "non-finite", "few finite rows", "huge", "tiny", "equal rows"])
def test_general_data(case, dtype):
    """The matrix form's hard data with enough queries that it is the form that runs."""
    with np.errstate(over="ignore", under="ignore"):
        x, y = matrix_data(case, dtype, np.random.default_rng(5))
    ix = S.Index(x)
    many = ix.knn(np.tile(y, (1024 // len(y) + 1, 1)), 9)
    oi, od, oc = O.linear_find_batch(x, y, 9)
    for r in range(0, len(many[2]), 13):
        c = int(oc[r % len(y)])
        assert many[2][r] == c
        np.testing.assert_array_equal(many[0][r, :c], oi[r % len(y), :c])
        np.testing.assert_array_equal(many[1][r, :c].view(np.uint64), od[r % len(y), :c].view(np.uint64))
