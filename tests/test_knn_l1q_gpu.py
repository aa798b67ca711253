"""Coded Manhattan kNN against the oracle: indices in heap-array order and
distance bits must be equal.  Sizes at the edges of the tiles, chunks, query
tilings (up to 32 queries, 128 per tile) and levels; data that clamp, leave
the code's range or come in an unfavourable order."""
import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu


def check(x, q, k):
    gi, gd, gc = S.Index(x).knn(q, k, S.SC_MANHATTAN, 1, S.SC_MIXED)
    oi, od, oc = O.linear_find_batch(x, q, k, O.MANHATTAN)
    np.testing.assert_array_equal(gc, oc)
    for r in range(q.shape[0]):
        c = int(oc[r])
        np.testing.assert_array_equal(gi[r, :c], oi[r, :c], err_msg=f"query {r}")
        np.testing.assert_array_equal(gd[r, :c].view(np.uint64), od[r, :c].view(np.uint64))


@pytest.mark.parametrize("n,q,d,k", [
    (1, 1, 1, 1), (127, 32, 2, 64), (128, 33, 15, 5), (1023, 128, 16, 10), (1025, 129, 17, 1),
    (1153, 3, 31, 20), (17_000, 32, 48, 9), (17_000, 33, 47, 64), (40_001, 1, 100, 3),
    (30_000, 260, 20, 16), (2_500, 5, 900, 4)])
def test_sizes(n, q, d, k):
    rng = np.random.default_rng(n + q)
    check(rng.normal(size=(n, d)).astype(np.float32), rng.normal(size=(q, d)).astype(np.float32), k)


@pytest.mark.parametrize("q", [20, 150])
@pytest.mark.parametrize("case", ["integers", "sorted by class", "approaching", "far queries",
                                  "non-finite queries", "wide range", "equal rows"])
def test_data(case, q):
    rng = np.random.default_rng(11)
    n, d = 6_000, 10
    x, qs = rng.normal(size=(n, d)), rng.normal(size=(q, d))
    if case == "integers":  # ties
        x, qs = np.rint(2 * x), np.rint(2 * qs)
    elif case == "sorted by class":
        lab = np.sort(rng.integers(0, 5, n))
        centres = rng.normal(0, 20, size=(5, d))
        x, qs = x + centres[lab], qs + centres[rng.integers(0, 5, q)]
    elif case == "approaching":
        x, qs = np.linspace(30, 1, n)[:, None] * np.ones((1, d)), 0.01 * qs
    elif case == "far queries":  # clamped codes
        qs = qs * 100
    elif case == "non-finite queries":
        qs[3, 1], qs[7, 2] = np.nan, np.inf
    elif case == "wide range":  # declined: the f32 scan answers
        x[5] *= 1e6
    elif case == "equal rows":
        x[:] = x[0]
    check(x.astype(np.float32), qs.astype(np.float32), 7)
