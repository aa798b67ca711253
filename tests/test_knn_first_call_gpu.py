"""The first plain Euclidian search of an index prepares its norms: it has to return before its stream
gets there, and neither may searches on other streams wait for it."""
import ctypes as C

import numpy as np
import pytest

from smartcore_amd import _capi as S

pytestmark = pytest.mark.gpu

N, D, Q, K = 100_000, 24, 300, 7
BUSY = 4 << 30  # bytes filled to keep a stream busy, about a millisecond each time
NOT_READY = 600


class Hip:
    def __init__(self):
        S.lib()
        self.L = C.CDLL("libamdhip64.so.7")
        self.L.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.L.hipFree.argtypes = [C.c_void_p]
        self.L.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
        self.L.hipMemsetAsync.argtypes = [C.c_void_p, C.c_int, C.c_size_t, C.c_void_p]
        self.L.hipStreamCreateWithFlags.argtypes = [C.POINTER(C.c_void_p), C.c_uint]
        for f in ("hipStreamQuery", "hipStreamSynchronize", "hipStreamDestroy"):
            getattr(self.L, f).argtypes = [C.c_void_p]

    def malloc(self, nbytes):
        p = C.c_void_p()
        assert self.L.hipMalloc(C.byref(p), nbytes) == 0
        return p

    def stream(self):
        s = C.c_void_p()
        assert self.L.hipStreamCreateWithFlags(C.byref(s), 1) == 0  # non-blocking
        return s


@pytest.fixture(scope="module")
def setting():
    hip = Hip()
    rng = np.random.default_rng(4)
    x, y = rng.normal(size=(N, D)).astype(np.float32), rng.normal(size=(Q, D)).astype(np.float32)
    want = S.Index(x).knn(y, K)
    dy = hip.malloc(y.nbytes)
    assert hip.L.hipMemcpy(dy, y.ctypes.data, y.nbytes, 1) == 0
    fill, streams = hip.malloc(BUSY), [hip.stream(), hip.stream()]
    yield hip, x, want, dy, fill, streams
    for s in streams:
        hip.L.hipStreamSynchronize(s)
        hip.L.hipStreamDestroy(s)
    hip.L.hipFree(fill)
    hip.L.hipFree(dy)


def search(hip, ix, dy, s):
    out = [hip.malloc(Q * K * 8), hip.malloc(Q * K * 8), hip.malloc(Q * 4)]
    ix.knn_device(dy.value, Q, K, *(p.value for p in out), stream=s.value)
    return out


def check(hip, out, want):
    for p, w in zip(out, want):
        w = np.ascontiguousarray(w)
        got = np.empty_like(w)
        assert hip.L.hipMemcpy(got.ctypes.data, p, w.nbytes, 2) == 0
        hip.L.hipFree(p)
        np.testing.assert_array_equal(got.view(np.uint8), w.view(np.uint8))


def test_first_call_does_not_wait(setting):
    hip, x, want, dy, fill, (a, b) = setting
    warm = S.Index(x)
    for s in (a, b):  # streams, scratch and kernels in place
        out = search(hip, warm, dy, s)
        assert hip.L.hipStreamSynchronize(s) == 0
        check(hip, out, want)
    ix = S.Index(x)
    for _ in range(150):
        assert hip.L.hipMemsetAsync(fill, 1, BUSY, a) == 0
    first = search(hip, ix, dy, a)
    assert hip.L.hipStreamQuery(a) == NOT_READY
    second = search(hip, ix, dy, b)  # the first stream's norms are not there yet
    assert hip.L.hipStreamSynchronize(b) == 0
    assert hip.L.hipStreamQuery(a) == NOT_READY
    again = search(hip, ix, dy, a)
    check(hip, second, want)
    assert hip.L.hipStreamSynchronize(a) == 0
    check(hip, first, want)
    check(hip, again, want)
    third = search(hip, ix, dy, b)
    assert hip.L.hipStreamSynchronize(b) == 0
    check(hip, third, want)
