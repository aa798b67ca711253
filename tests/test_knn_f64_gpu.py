"""FP64 matrix-core kNN (Euclidian, plain form) against the oracle: indices in
heap-array order and distance bits must be equal, so no tolerance enters.
The sizes sit at the edges of the 128 x 128 tile, the 16-dimension chunk, the
1,024-row dense prefix and the level split; the data cases are the ones a
bound could get wrong."""
import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu


def check(x, q, k):
    gi, gd, gc = S.Index(x).knn(q, k)
    oi, od, oc = O.linear_find_batch(x, q, k)
    np.testing.assert_array_equal(gc, oc)
    for r in range(q.shape[0]):
        c = int(oc[r])
        np.testing.assert_array_equal(gi[r, :c], oi[r, :c], err_msg=f"query {r}")
        np.testing.assert_array_equal(gd[r, :c].view(np.uint64), od[r, :c].view(np.uint64))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,q,d,k", [
    (1, 1, 1, 1), (64, 3, 3, 64), (127, 128, 4, 5), (129, 129, 5, 1), (1023, 2, 16, 33),
    (1024, 127, 17, 10), (1025, 130, 15, 64), (1153, 256, 31, 7), (4000, 65, 33, 20),
    (17_501, 140, 20, 10), (40_001, 1, 100, 3), (30_000, 33, 130, 16)])
def test_sizes(n, q, d, k, dtype):
    rng = np.random.default_rng(n * 7 + q)
    check(rng.normal(size=(n, d)).astype(dtype), rng.normal(size=(q, d)).astype(dtype), k)


def _data(case, dtype, rng):
    n, d, q = 6_000, 12, 40
    x, qs = rng.normal(size=(n, d)), rng.normal(size=(q, d))
    if case == "sorted by class":  # the prefix holds one class only
        lab = np.sort(rng.integers(0, 6, n))
        centres = rng.normal(0, 30.0, size=(6, d))
        x, qs = centres[lab] + x, centres[rng.integers(0, 6, q)] + qs
    elif case == "approaching":  # every row is an entrant: lists overflow
        x = np.linspace(50.0, 1.0, n)[:, None] * np.ones((1, d))
        qs = 0.01 * qs
    elif case == "ties":
        x, qs = np.rint(x), np.rint(qs)
    elif case == "far from the origin":
        x, qs = x + 1e6, qs + 1e6
    elif case == "non-finite":
        x[rng.random(n) < 0.1, 3] = np.nan
        x[rng.random(n) < 0.1, 5] = np.inf
        qs[3, 2], qs[7, 0] = np.nan, -np.inf
    elif case == "few finite rows":
        x[3:, 1] = np.nan
    elif case == "huge":  # squared norms past the bound's range (f64) / f32 overflow
        big = 1e200 if dtype == np.float64 else 1e30
        x[::7] *= big
        qs[::5] *= big
        x[35] = qs[5]
    elif case == "tiny":  # squares underflow
        s = 1e-170 if dtype == np.float64 else 1e-25
        x, qs = x * s, qs * s
    elif case == "equal rows":
        x[:] = x[0]
    return x.astype(dtype), qs.astype(dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", ["sorted by class", "approaching", "ties", "far from the origin",
                                  "non-finite", "few finite rows", "huge", "tiny", "equal rows"])
def test_data(case, dtype):
    with np.errstate(over="ignore", under="ignore"):
        x, q = _data(case, dtype, np.random.default_rng(5))
    check(x, q, 9)


def test_rows_sorted_by_class_stay_off_the_sequential_kernel():
    rng = np.random.default_rng(9)
    lab = np.sort(rng.integers(0, 8, 60_000))
    centres = rng.normal(0, 30.0, size=(8, 16))
    x = centres[lab] + rng.normal(size=(60_000, 16))
    q = centres[rng.integers(0, 8, 600)] + rng.normal(size=(600, 16))
    S.Index(x).knn(q, 10)
    assert S.last_stats()["overflow_queries"] == 0
