"""Searches of an index that leaves no room for what the FP64 matrix form keeps beside the rows (eight
bytes each): they have to answer, as they do without that form."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu

LEFT = 1_400_000_000  # bytes of device memory that stay free


@pytest.fixture
def nearly_full():
    """350,000,000 rows on the device (their norms: 2.8 GB) and the rest of the memory taken but LEFT."""
    n = 350_000_000
    x = np.random.default_rng(6).random((n, 1), dtype=np.float32)
    x += 50.0
    x[[3, 77, n // 2, n - 1], 0] = [0.75, 0.25, 0.5, 1.25]
    ix = S.Index(x)
    hip = C.CDLL("libamdhip64.so.7")
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipFree.argtypes = [C.c_void_p]
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
    free, total, held = C.c_size_t(), C.c_size_t(), []
    while True:
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        if free.value < LEFT + (1 << 28):
            break
        p = C.c_void_p()
        if hip.hipMalloc(C.byref(p), min(16 << 30, free.value - LEFT)) != 0:
            break
        held.append(p)
    yield x, ix
    for p in held:
        hip.hipFree(p)


def test_searches_without_room_for_norms(nearly_full):
    x, ix = nearly_full
    y = np.zeros((1, 1), np.float32)
    gi, gd, gc = ix.knn(y, 3)
    oi, od = O.linear_find(x, y[0], 3)
    assert gc[0] == 3 and S.last_stats()["overflow_queries"] == 1  # by the sequential kernel
    np.testing.assert_array_equal(gi[0], oi)
    np.testing.assert_array_equal(gd[0].view(np.uint64), np.asarray(od).view(np.uint64))
    (rows, dist), = ix.radius(y, 1.0)
    oi, od = O.linear_find_radius(x, y[0], 1.0, O.EUCLIDIAN)
    np.testing.assert_array_equal(rows, oi)
    np.testing.assert_array_equal(dist.view(np.uint64), od.view(np.uint64))
