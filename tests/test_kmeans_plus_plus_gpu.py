"""k-means++ rounds that the host has to decide: a cutoff on the boundary between two rows, and costs
whose sum is not finite; labels against the oracle, and how many rounds were launched."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu


def labels_and_launches(x, k, seed):
    L = S.lib()
    L.sc_profile_enable.argtypes = [C.c_int]
    L.sc_profile_read.argtypes = [C.c_char_p, C.POINTER(C.c_double), C.POINTER(C.c_uint64)]
    ix, ms, rounds = S.Index(x), C.c_double(), C.c_uint64()
    L.sc_profile_enable(1)
    try:
        y = ix.kmeans_plus_plus(k, seed)
        L.sc_profile_read(b"kmeanspp_round", C.byref(ms), C.byref(rounds))
    finally:
        L.sc_profile_enable(0)
    return y, rounds.value


def boundary_seed(n, other):
    """A seed whose second draw puts the cutoff within the bound of a boundary between two of `other`
    rows at distance 1 (the rest are copies of the first centre)."""
    delta = 4.0 * (n + 64.0) * 2.0 ** -53 * other
    for seed in range(200_000):
        r = O.SmallRng(seed)
        r.gen_range(n)
        cut = r.gen_f64() * other
        if abs(cut - round(cut)) < 0.5 * delta and 1 < cut < other - 1:
            return seed
    raise AssertionError("no seed")


def test_cutoff_between_two_rows():
    n, k = 1_000_000, 12
    x = np.zeros((n, 1))
    x[1::2] = 1.0
    seed = boundary_seed(n, n // 2)
    y, rounds = labels_and_launches(x, k, seed)
    assert rounds > k  # the first round went to the host, the others were queued again
    np.testing.assert_array_equal(y, O.kmeans_plus_plus(x, k, seed))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("bad", [2, 40])
def test_costs_without_a_finite_sum(bad, dtype):
    rng = np.random.default_rng(8)
    n, k = 3_000, 64
    x = rng.normal(size=(n, 5)).astype(dtype)
    x[rng.choice(n, bad, replace=False), 2] = np.nan
    for seed in (None, 5, 77):
        y, rounds = labels_and_launches(x, k, seed)
        np.testing.assert_array_equal(y, O.kmeans_plus_plus(x, k, seed))
        assert rounds <= 2 * k


def test_sum_becomes_finite():
    """Distances that overflow until a centre is near: the host decides first, the device after."""
    rng = np.random.default_rng(9)
    x = rng.normal(size=(4_000, 3))
    x[::2] *= 1e-3
    x[1::2] += 1e200
    k = 40
    for seed in (None, 3, 11):
        y, rounds = labels_and_launches(x, k, seed)
        np.testing.assert_array_equal(y, O.kmeans_plus_plus(x, k, seed))
        assert rounds <= 2 * k
