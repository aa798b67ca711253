"""The rescoring of a query's candidates with 512 threads (up to 512 queries, narrow rows) and with
128, against the oracle: rows sorted by class, whose first rows bound the others badly, so that a
query has several batches of candidates; and ordinary rows, a few hundred of them.  Indices in heap
order and distance bits."""
import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu


def check(x, y, k, metric, om, mode):
    gi, gd, gc = S.Index(x).knn(y, k, metric, 3, mode)
    per_query = S.last_stats()["candidates"] / len(y)
    oi, od, oc = O.linear_find_batch(x, y, k, om, 3)
    np.testing.assert_array_equal(gc, oc)
    for r in range(len(y)):
        c = int(oc[r])
        np.testing.assert_array_equal(gi[r, :c], oi[r, :c])
        np.testing.assert_array_equal(gd[r, :c].view(np.uint64), od[r, :c].view(np.uint64))
    return per_query


@pytest.mark.parametrize("form", ["plain64", "plain32", "manhattan"])
@pytest.mark.parametrize("n,q,d,k,classes", [(70_000, 1, 5, 3, 6), (66_001, 511, 3, 64, 1), (66_001, 513, 3, 1, 6),
                                             (70_000, 20, 32, 10, 6), (40_000, 2, 1_100, 10, 1),
                                             (1_500, 512, 7, 64, 6)])
def test_finish(n, q, d, k, classes, form):
    if form == "manhattan" and d > 832:
        pytest.skip("no codes at this width")
    rng = np.random.default_rng(n + q + d)
    centre = 30 * rng.normal(size=(classes, d))
    x = rng.normal(size=(n, d)) + centre[np.sort(rng.integers(0, classes, size=n))]
    y = rng.normal(size=(q, d)) + centre[-1]
    dtype = np.float64 if form == "plain64" else np.float32
    x, y = x.astype(dtype), y.astype(dtype)
    if form == "manhattan":
        seen = check(x, y, k, S.SC_MANHATTAN, O.MANHATTAN, S.SC_MIXED)
    else:
        seen = check(x, y, k, S.SC_EUCLIDIAN, O.EUCLIDIAN, S.SC_PLAIN_FP64)
    if classes > 1 and q <= 20:
        assert seen > 1_024  # more than a batch
