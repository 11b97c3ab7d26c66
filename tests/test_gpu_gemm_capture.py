"""Products that are split along k when they run directly (few tiles, a long k), recorded into a
HIP graph on the caller's stream: a recorded call takes no pool scratch, so replays between other
calls give the direct call's result.  Small integers: every sum is exact in any order."""
import ctypes

import numpy as np
import pytest

from _devmem import Matrix

pytestmark = pytest.mark.gpu
VP, CI = ctypes.c_void_p, ctypes.c_int


@pytest.fixture(scope="module")
def hip():
    h = ctypes.CDLL("libamdhip64.so")
    h.hipStreamCreate.argtypes = [ctypes.POINTER(VP)]
    h.hipStreamBeginCapture.argtypes = [VP, CI]
    h.hipStreamEndCapture.argtypes = [VP, ctypes.POINTER(VP)]
    h.hipGraphInstantiate.argtypes = [ctypes.POINTER(VP), VP, VP, VP, ctypes.c_size_t]
    h.hipGraphLaunch.argtypes = [VP, VP]
    for f in (h.hipStreamSynchronize, h.hipStreamDestroy, h.hipGraphDestroy, h.hipGraphExecDestroy):
        f.argtypes = [VP]
    return h


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("m,n,k", [(64, 64, 2048), (33, 70, 1031), (128, 32, 512)])
def test_recorded_product(gpu, hip, prec, m, n, k):
    lib = gpu.library()
    f, real, dt = ((lib.gpublas_dev_dgemm, ctypes.c_double, np.float64) if prec == "d" else
                   (lib.gpublas_dev_sgemm, ctypes.c_float, np.float32))
    rng = np.random.default_rng(m + k)
    a, b = (rng.integers(-3, 4, s).astype(dt) for s in ((m, k), (k, n)))
    A, B, C, D = (Matrix(gpu, x) for x in (a, b, np.zeros((m, n), dt), np.zeros((m, n), dt)))

    def call(stream, out):
        return f(stream, ctypes.c_char(b"N"), ctypes.c_char(b"N"), CI(m), CI(n), CI(k), real(1.0),
                 VP(A.ptr), CI(m), VP(B.ptr), CI(k), real(0.0), VP(out.ptr), CI(m))

    s, graph, run = VP(), VP(), VP()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    assert hip.hipStreamBeginCapture(s, 0) == 0
    err = call(s, C)
    assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0 and err == 0
    assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, 0) == 0
    want = a @ b
    for rep in range(3):
        C.put(np.full((m, n), rep + 0.5))
        assert hip.hipGraphLaunch(run, s) == 0
        assert call(s, D) == 0  # directly, with scratch, between the replays
        assert hip.hipStreamSynchronize(s) == 0
        assert np.array_equal(C.get(), want) and np.array_equal(D.get(), want)
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    assert hip.hipStreamDestroy(s) == 0
    for x in (A, B, C, D):
        x.free()
