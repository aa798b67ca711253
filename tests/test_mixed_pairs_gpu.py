"""Mixed Euclidian kNN with more candidates in one pair of lists than a level's workgroup merges at a
time (1,024): the replay merges the pair; no query may go to the sequential kernel."""
import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first,second", [(400, 400), (456, 456), (650, 650), (690, 290), (250, 690)])
def test_long_pairs(first, second):
    """66,048 queries of 600,000 rows in two segments: 800 entries a half for rows 16,384 .. 131,071.
    So many rows of each half of the first segment's tiles, and about 56 of its other rows, are closer
    than the 32nd of the rows before them."""
    rng = np.random.default_rng(first)
    n, q, d, k = 600_000, 66_048, 16, 32
    x = (10.0 * rng.normal(size=(n, d))).astype(np.float32)
    rows = np.arange(16_384, 16_384 + 57_344)
    half = (rows >> 2) & 1
    pick = np.concatenate([rng.choice(rows[half == 0], first, replace=False),
                           rng.choice(rows[half == 1], second, replace=False)])
    x[pick] = (0.2 * rng.normal(size=(len(pick), d))).astype(np.float32)
    x[pick[::5]] = x[pick[0]]  # equal distances: the order decides
    y = (0.05 * rng.normal(size=(q, d))).astype(np.float32)
    ix = S.Index(x)
    gi, gd, gc = ix.knn(y, k, S.SC_EUCLIDIAN, 2, S.SC_MIXED)
    stats = S.last_stats()
    assert stats["overflow_queries"] == 0 and stats["candidates"] >= q * len(pick)
    pi, pd, pc = ix.knn(y, k)
    np.testing.assert_array_equal(gc, pc)
    np.testing.assert_array_equal(gi, pi)
    np.testing.assert_array_equal(gd.view(np.uint64), pd.view(np.uint64))
    for r in (0, q - 1):
        oi, od = O.linear_find(x, y[r], k)
        np.testing.assert_array_equal(gi[r], oi)
        np.testing.assert_array_equal(gd[r].view(np.uint64), np.asarray(od).view(np.uint64))
