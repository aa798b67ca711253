"""Euclidian radius searches whose candidate lists overflow, and the capped pass of the other metrics:
against the same queries searched in sets so small (up to 3,500,000 pairs) that the count and fill
passes answer, and against the oracle; lists and distance bits."""
import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu


def same(got, want):
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[1].view(np.uint64), want[1].view(np.uint64))


def check(x, q, radius, pick, metric=S.SC_EUCLIDIAN, om=O.EUCLIDIAN):
    ix = S.Index(x)
    got = ix.radius(q, radius, metric)
    small = max(1, 3_500_000 // len(x))
    for a in range(0, len(pick), small):
        for i, ref in zip(pick[a:a + small], ix.radius(q[pick[a:a + small]], radius, metric)):
            same(got[i], ref)
    for i in pick[:: max(1, len(pick) // 5)]:
        same(got[i], O.linear_find_radius(x, q[i], radius, om))
    return np.array([len(g[0]) for g in got])


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_lists_overflow(dtype):
    """20,000 queries x 60,000 rows: five lists of 671 entries a query.  Queries in the row blocks of
    2,500 and 9,000 overflow and are swept again; a norm out of the bound's range takes the two
    passes."""
    rng = np.random.default_rng(31)
    n, q, d = 60_000, 20_000, 4
    x, y = rng.normal(0, 6, size=(n, d)), rng.normal(0, 6, size=(q, d))
    x[20_000:22_500] = 40 + 0.1 * rng.normal(size=(2_500, d))
    x[30_000:39_000] = -40 + 0.1 * rng.normal(size=(9_000, d))
    y[100:1_100] = 40 + 0.1 * rng.normal(size=(1_000, d))
    y[1_500:1_600] = -40 + 0.1 * rng.normal(size=(100, d))
    y[5] = 1e150 if dtype == np.float64 else 1e20
    x[7] = y[5]
    with np.errstate(over="ignore"):
        x, y = x.astype(dtype), y.astype(dtype)
    pick = np.concatenate([[5], np.arange(100, 400), np.arange(1_500, 1_550), rng.choice(q, 400, replace=False)])
    counts = check(x, y, 1.2, pick)
    assert counts[100:1_100].min() > 671 and counts[1_500:1_600].min() > 5 * 671 and counts[2_000:].max() < 671


def test_no_list_holds_a_query():
    """Every query's norm is out of the bound's range: nothing comes from the sweep."""
    rng = np.random.default_rng(2)
    x = 1e150 * rng.normal(size=(9_000, 3))
    check(x, x[:400], 1e149, np.arange(0, 400, 3))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("q,share", [(40, 0.02), (40, 0.3), (1_000, 0.01), (129, 0.15)])
def test_many_matches(q, share, dtype):
    rng = np.random.default_rng(q)
    x, y = rng.normal(size=(100_000, 3)).astype(dtype), rng.normal(size=(q, 3)).astype(dtype)
    radius = float(np.quantile(np.sqrt(((x[:20_000] - y[0].astype(np.float64)) ** 2).sum(1)), share))
    counts = check(x, y, radius, np.arange(0, q, max(1, q // 60)))
    assert counts[0] > 0.5 * share * len(x)


def test_distances_on_the_radius():
    """A grid: a query's matches lie on the radius itself by the hundred, so no bound decides them."""
    rng = np.random.default_rng(3)
    x, y = rng.integers(0, 12, size=(50_000, 3)).astype(np.float64), rng.integers(0, 12, size=(300, 3)).astype(np.float64)
    for radius in (5.0, np.nextafter(5.0, 0)):
        check(x, y, float(radius), np.arange(0, 300, 7))


def test_capped_pass_of_the_manhattan_metric():
    """140,000 queries: every query block scans all rows, a query's matches go to a slot of 256 entries
    and the queries with more are searched again."""
    rng = np.random.default_rng(61)
    n, d = 140_000, 8
    x = rng.normal(0.0, 4.0, size=(n, d))
    x[:3_000] = rng.normal(0.0, 0.3, size=(3_000, d))
    pick = np.concatenate([np.arange(0, 300), rng.choice(n, 500, replace=False)])
    counts = check(x, x, 2.2, pick, S.SC_MANHATTAN, O.MANHATTAN)
    assert 0 < (counts > 256).sum() < n and (counts <= 256).sum() > 0
