"""DBSCAN over enough rows to be put in groups first (32,768): copies of one small set, far apart or
on top of each other, against the oracle on that set.  The values are multiples of 2^-10 and the
shifts whole numbers, so every difference and square of near rows is exact in either type and a
copy's neighbours are the set's own."""
import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu

COPIES = 24


def core_rows(x, eps, ms):
    x = x.astype(np.float64)
    near = np.zeros(len(x), np.int64)
    for i in range(len(x)):
        with np.errstate(invalid="ignore"):
            near[i] = np.count_nonzero(np.sqrt(((x - x[i]) ** 2).sum(1)) <= eps)
    return near >= ms


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", ["apart", "non-finite", "wide", "together"])
def test_grouped_fit(case, dtype):
    rng = np.random.default_rng(23)
    m, d, eps, ms = 1500, 3, 0.35, 6
    if case == "wide":  # more values than the grouping looks at
        m, d, eps = 1400, 70, 0.75
    x = rng.normal(size=(m, d))
    if case == "wide":
        x *= 0.08
    x = np.rint(1024 * x) / 1024
    if case == "non-finite":
        x[::7, 1], x[3::13, 0] = np.nan, np.inf
    x = x.astype(dtype)
    lab, _ = O.dbscan_fit(x, eps, ms)
    lab = np.asarray(lab)
    core = core_rows(x, eps, ms)
    n = m * COPIES  # row i of copy b is row i COPIES + b
    if case == "together":
        rows, want, count, ms = np.repeat(x, COPIES, axis=0), np.repeat(lab, COPIES), lab.max() + 1, ms * COPIES
    else:
        shift = np.zeros((COPIES, d), dtype)
        shift[:, 0] = 64 * np.arange(COPIES)
        rows = (x[:, None, :] + shift[None]).reshape(n, d)
        # clusters by their smallest core row
        first = {}
        for i in np.flatnonzero(core):
            first.setdefault(lab[i], i)
        order = sorted((i * COPIES + b, b, c) for c, i in first.items() for b in range(COPIES))
        number = {(b, c): k for k, (_, b, c) in enumerate(order)}
        want = np.array([number.get((b, lab[i]), -1) for i in range(m) for b in range(COPIES)])
        count = len(order)
    assert n >= 32768 and count > 0 and (want < 0).any()
    got, nc = S.Index(rows).dbscan_fit(eps, ms)
    assert nc == count
    np.testing.assert_array_equal(got, want)
