"""Euclidian radius search and DBSCAN on the FP64 matrix form against the
oracle: lists, distance bits, labels and cluster counts must be equal."""
import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu


def check(x, q, radius, every=1):
    got = S.Index(x).radius(q, radius)
    for i in range(0, q.shape[0], every):
        oi, od = O.linear_find_radius(x, q[i], radius, O.EUCLIDIAN)
        np.testing.assert_array_equal(got[i][0], oi, err_msg=f"query {i}")
        np.testing.assert_array_equal(got[i][1].view(np.uint64), od.view(np.uint64))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,q,d", [(1, 1, 1), (127, 130, 3), (128, 128, 16), (129, 1, 17),
                                   (3000, 257, 5), (20_011, 140, 33), (90_000, 3, 8)])
def test_radius_sizes(n, q, d, dtype):
    rng = np.random.default_rng(n + q)
    x, qs = rng.normal(size=(n, d)).astype(dtype), rng.normal(size=(q, d)).astype(dtype)
    radius = float(np.quantile(np.sqrt(((x[:500] - qs[0]) ** 2).sum(1)), 0.05)) + 1e-3
    check(x, qs, radius, every=max(1, q // 40))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", ["grid", "non-finite", "huge", "tiny", "clustered order", "infinite radius"])
def test_radius_data(case, dtype):
    rng = np.random.default_rng(8)
    x, q = rng.normal(size=(4000, 6)), rng.normal(size=(50, 6))
    radius = 1.5
    if case == "grid":  # many distances equal to the radius
        x, q, radius = np.rint(2 * x), np.rint(2 * q), 3.0
    elif case == "non-finite":
        x[::9, 2], x[5::11, 0], q[3, 1], q[4, 4] = np.nan, np.inf, np.nan, -np.inf
    elif case == "huge":
        big = 1e200 if dtype == np.float64 else 1e25
        x[::5] *= big
        q[:10] = x[:50:5]
    elif case == "tiny":
        s = 1e-160 if dtype == np.float64 else 1e-22
        x, q, radius = x * s, q * s, radius * s
    elif case == "clustered order":  # a query's matches sit together: lists overflow
        x = np.repeat(rng.normal(0, 20, size=(4, 6)), 5000, axis=0) + 0.1 * rng.normal(size=(20_000, 6))
        q = x[::2500]
    elif case == "infinite radius":
        x[7, 1], radius = np.inf, float("inf")
    with np.errstate(over="ignore", under="ignore"):
        x, q = x.astype(dtype), q.astype(dtype)
    check(x, q, radius)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", ["one row", "tile edge", "duplicates", "non-finite", "dense"])
def test_dbscan_data(case, dtype):
    rng = np.random.default_rng(17)
    x, eps, ms = rng.normal(size=(1500, 3)), 0.35, 6
    if case == "one row":
        x, ms = x[:1], 1
    elif case == "tile edge":
        x = x[:257]
    elif case == "duplicates":
        x = np.rint(3 * x) / 3
    elif case == "non-finite":
        x[::7, 1], x[3::13, 0] = np.nan, np.inf
    elif case == "dense":  # more pairs than the first store holds
        x, eps = 0.01 * rng.normal(size=(8_500, 2)), 1.0
        x[::1000] += 5.0
    x = x.astype(dtype)
    lab, nc = S.Index(x).dbscan_fit(eps, ms)
    olab, onc = O.dbscan_fit(x, eps, ms)
    assert nc == onc
    np.testing.assert_array_equal(lab, olab)
