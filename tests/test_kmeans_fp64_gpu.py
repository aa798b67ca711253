"""FP64 k-means: the one-thread-per-row assignment, the sorted block sums and
k-means++ on the device, at the edges of their rules.  Labels are compared
with the oracle's; sums bit for bit with the fixed order (rows in row order
inside blocks of 2,048, blocks in order, up to sixteen of them) computed by
sequential numpy sums."""
import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu


def ordered_sums(x, labels, k):
    out = np.zeros((k, x.shape[1]))
    for b in range(0, x.shape[0], 2048):
        xb, lb = x[b:b + 2048].astype(np.float64), labels[b:b + 2048]
        part = np.zeros_like(out)
        for c in range(k):
            rows = xb[lb == c]
            if len(rows):
                part[c] = np.cumsum(np.concatenate([np.zeros((1, x.shape[1])), rows]), axis=0)[-1]
        out = out + part
    return out


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,d,k", [
    (1, 1, 1), (2048, 16, 32), (2049, 17, 33), (5000, 32, 2), (4097, 33, 10), (3000, 48, 5),
    (3000, 49, 32), (3000, 64, 33), (2500, 65, 128), (2500, 9, 129), (1500, 130, 7)])
def test_step(n, d, k, dtype):
    rng = np.random.default_rng(n + d + k)
    x = (rng.normal(0, 5, size=(max(k, 2), d))[rng.integers(0, max(k, 2), n)] + rng.normal(size=(n, d))).astype(dtype)
    c = x[rng.integers(0, n, k)].astype(np.float64) + 0.01 * rng.normal(size=(k, d))
    dist, sums, counts, memb = S.Index(x).kmeans_step(c)
    _, _, ocounts, omemb = O.lloyd_step_brute(x, c)
    np.testing.assert_array_equal(memb, omemb)
    np.testing.assert_array_equal(counts, ocounts)
    np.testing.assert_array_equal(sums, ordered_sums(x, memb, k))
    np.testing.assert_array_equal(S.kmeans_predict(x, c), omemb)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_assignment_rule_on_ties_and_non_finite_rows(dtype):
    rng = np.random.default_rng(4)
    x = np.rint(rng.normal(size=(70_000, 5))).astype(dtype)
    x[5, 1], x[9, 2] = np.nan, np.inf
    c = np.rint(rng.normal(size=(7, 5)))
    c[4] = c[2]
    c[6] = np.nan
    np.testing.assert_array_equal(S.kmeans_predict(x, c), O.kmeans_predict(x, c))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", ["small", "blocks", "equal rows", "non-finite", "k = n"])
def test_kmeans_plus_plus(case, dtype):
    rng = np.random.default_rng(6)
    n, d, k = {"small": (100, 2, 5), "k = n": (40, 3, 40)}.get(case, (30_001, 6, 9))
    x = rng.normal(size=(n, d)).astype(dtype)
    if case == "equal rows":
        x[:] = x[0]
        x[20_000:] += 1
    elif case == "non-finite":  # the distances' sum overflows: the host decides
        x[[3, 900, 1500], 1] = np.nan
        x[77, 0] = np.inf
    ix = S.Index(x)
    for seed in (None, 0, 3, 12345):
        np.testing.assert_array_equal(ix.kmeans_plus_plus(k, seed), O.kmeans_plus_plus(x, k, seed))
