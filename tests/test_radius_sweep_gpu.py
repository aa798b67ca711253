"""Euclidian radius searches on both sides of the line between the two passes and the FP64 matrix
sweep (3,500,000 pairs): against the oracle on some of the queries, lists and distance bits."""
import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", ["plain", "grid", "non-finite", "huge", "tiny", "clustered order"])
@pytest.mark.parametrize("n,q,d", [(3500, 1000, 3), (3500, 1001, 3), (38_401, 92, 17), (28_000, 129, 33)])
def test_sweep(n, q, d, case, dtype):
    rng = np.random.default_rng(n + q)
    x, y = rng.normal(size=(n, d)), rng.normal(size=(q, d))
    y[:5] = x[:5]
    radius = {3: 0.4, 17: 3.4, 33: 5.8}[d]
    if case == "grid":  # distances on the radius itself
        x, y, radius = np.rint(2 * x) / 2, np.rint(2 * y) / 2, np.round(radius) or 0.5
    elif case == "non-finite":
        x[::7, 1], x[3::13, 0], y[1, 0], y[2, 2] = np.nan, np.inf, np.nan, -np.inf
    elif case == "huge":
        big = 1e200 if dtype == np.float64 else 1e25
        x[::5] *= big
        y[:3] *= big
    elif case == "tiny":
        s = 1e-160 if dtype == np.float64 else 1e-22
        x, y, radius = x * s, y * s, radius * s
    elif case == "clustered order":  # a query's matches sit together: lists overflow
        x[n // 3:n // 3 + 3000] = x[0] + 1e-3 * x[n // 3:n // 3 + 3000]
    with np.errstate(over="ignore", under="ignore"):
        x, y = x.astype(dtype), y.astype(dtype)
    got = S.Index(x).radius(y, radius)
    for i in list(range(6)) + [q // 2, q - 1]:
        oi, od = O.linear_find_radius(x, y[i], radius, O.EUCLIDIAN)
        np.testing.assert_array_equal(got[i][0], oi, err_msg=f"query {i}")
        np.testing.assert_array_equal(got[i][1].view(np.uint64), od.view(np.uint64))
