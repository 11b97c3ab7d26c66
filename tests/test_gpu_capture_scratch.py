"""Calls that work through scratch memory, recorded into HIP graphs on a caller's stream and on the
library's own: the scratch belongs to the graph, so replays give the direct call's result while
direct calls on another stream take scratch of the same size, and after the library's workspace has
grown; it returns to the pool with the last executable graph.  Integer data where products are
summed: exact in any order."""
import ctypes

import numpy as np
import pytest

from _devmem import Matrix

pytestmark = pytest.mark.gpu
VP, CI, CD = ctypes.c_void_p, ctypes.c_int, ctypes.c_double


def c(ch):
    return ctypes.c_char(ch.encode())


@pytest.fixture(scope="module")
def hip(gb):
    h = ctypes.CDLL("libamdhip64.so")
    h.hipStreamCreate.argtypes = [ctypes.POINTER(VP)]
    h.hipStreamBeginCapture.argtypes = [VP, CI]
    h.hipStreamEndCapture.argtypes = [VP, ctypes.POINTER(VP)]
    h.hipGraphInstantiate.argtypes = [ctypes.POINTER(VP), VP, VP, VP, ctypes.c_size_t]
    h.hipGraphLaunch.argtypes = [VP, VP]
    for f in (h.hipStreamSynchronize, h.hipStreamDestroy, h.hipGraphDestroy, h.hipGraphExecDestroy):
        f.argtypes = [VP]
    return h


# name: (shapes of the operands, the last one the output; the call)
CALLS = {
    "dgemv": ([(1500, 1500), (1500, 1), (1500, 1)], lambda L, s, a, x, y: L.gpublas_dev_dgemv(
        s, c("N"), CI(1500), CI(1500), CD(1), a, CI(1500), x, CI(1), CD(0), y, CI(1))),
    "dsymv": ([(1500, 1500), (1500, 1), (1500, 1)], lambda L, s, a, x, y: L.gpublas_dev_dsymv(
        s, c("L"), CI(1500), CD(1), a, CI(1500), x, CI(1), CD(0), y, CI(1))),
    "dtrsv": ([(700, 700), (700, 1)], lambda L, s, a, x: L.gpublas_dev_dtrsv(
        s, c("L"), c("N"), c("N"), CI(700), a, CI(700), x, CI(1))),
    "dtrsv_strided": ([(300, 300), (600, 1)], lambda L, s, a, x: L.gpublas_dev_dtrsv(
        s, c("U"), c("T"), c("N"), CI(300), a, CI(300), x, CI(2))),
    "dtbmv": ([(9, 3000), (3000, 1)], lambda L, s, a, x: L.gpublas_dev_dtbmv(
        s, c("U"), c("N"), c("N"), CI(3000), CI(8), a, CI(9), x, CI(1))),
    "dgbmv": ([(21, 3000), (3000, 1), (3000, 1)], lambda L, s, a, x, y: L.gpublas_dev_dgbmv(
        s, c("N"), CI(3000), CI(3000), CI(10), CI(10), CD(1), a, CI(21), x, CI(1), CD(0), y, CI(1))),
    "dtrmm": ([(300, 300), (300, 200)], lambda L, s, a, b: L.gpublas_dev_dtrmm(
        s, c("L"), c("L"), c("N"), c("N"), CI(300), CI(200), CD(1), a, CI(300), b, CI(300))),
    "dsymm": ([(300, 300), (300, 200), (300, 200)], lambda L, s, a, b, o: L.gpublas_dev_dsymm(
        s, c("L"), c("U"), CI(300), CI(200), CD(1), a, CI(300), b, CI(300), CD(0), o, CI(300))),
    "zgemm": ([(200, 150), (300, 60), (200, 60)], lambda L, s, a, b, o: L.gpublas_dev_zgemm(
        s, c("N"), c("N"), CI(100), CI(60), CI(150), CD(1), CD(0), a, CI(100), b, CI(150), CD(0),
        CD(0), o, CI(100))),
}


def _operands(gpu, name, seed):
    rng = np.random.default_rng(seed)
    arrays = [rng.integers(-3, 4, s).astype(float) for s in CALLS[name][0]]
    if name.startswith("dtrsv"):
        np.fill_diagonal(arrays[0], 300.0 + seed)
    return [Matrix(gpu, a) for a in arrays]


def _record(hip, stream, call):
    graph, run = VP(), VP()
    assert hip.hipStreamBeginCapture(stream, 0) == 0
    err = call()
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0 and err == 0
    assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, 0) == 0
    assert hip.hipGraphDestroy(graph) == 0
    return run


@pytest.mark.parametrize("own", [False, True])
@pytest.mark.parametrize("name", list(CALLS))
def test_replays_beside_direct_calls(gpu, hip, name, own):
    lib, call = gpu.library(), CALLS[name][1]
    mine, other = VP(), VP()
    assert hip.hipStreamCreate(ctypes.byref(mine)) == 0 and hip.hipStreamCreate(ctypes.byref(other)) == 0
    recorded = VP(lib.gpublas_dev_stream()) if own else mine
    p, q = _operands(gpu, name, 1), _operands(gpu, name, 2)
    start = [m[-1].like.copy() for m in (p, q)]
    want = []
    for m in (p, q):
        assert call(lib, None, *(VP(x.ptr) for x in m)) == 0
        want.append(m[-1].get())
        m[-1].put(m[-1].like)
    run = _record(hip, recorded, lambda: call(lib, recorded, *(VP(x.ptr) for x in p)))
    big = Matrix(gpu, np.ones((4000, 4000)))
    vec = Matrix(gpu, np.ones((4000, 1)))
    try:
        for rep in range(5):
            p[-1].put(start[0])
            q[-1].put(start[1])
            if rep == 2:  # the library's workspace grows: the old one goes back to the pool
                assert lib.gpublas_dev_dsymv(None, c("L"), CI(4000), CD(1), VP(big.ptr), CI(4000),
                                             VP(vec.ptr), CI(1), CD(0), VP(vec.ptr), CI(1)) == 0
                vec.put(vec.like)
            assert hip.hipGraphLaunch(run, mine) == 0
            assert call(lib, other, *(VP(x.ptr) for x in q)) == 0
            assert hip.hipStreamSynchronize(mine) == 0 and hip.hipStreamSynchronize(other) == 0
            assert np.array_equal(p[-1].get(), want[0]), rep
            assert np.array_equal(q[-1].get(), want[1]), rep
    finally:
        assert hip.hipGraphExecDestroy(run) == 0
        for x in p + q + [big, vec]:
            x.free()
        assert hip.hipStreamDestroy(mine) == 0 and hip.hipStreamDestroy(other) == 0


def test_scratch_returns_with_the_graph(gpu, hip):
    lib, call = gpu.library(), CALLS["dtrmm"][1]
    lib.gpublas_dev_pool_bytes.restype = ctypes.c_size_t
    s = VP()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    m = _operands(gpu, "dtrmm", 1)

    def once():
        run = _record(hip, s, lambda: call(lib, s, *(VP(x.ptr) for x in m)))
        assert hip.hipGraphLaunch(run, s) == 0 and hip.hipStreamSynchronize(s) == 0
        assert hip.hipGraphExecDestroy(run) == 0

    once()
    held = lib.gpublas_dev_pool_bytes()
    for _ in range(8):
        once()
    assert lib.gpublas_dev_pool_bytes() == held
    for x in m:
        x.free()
    assert hip.hipStreamDestroy(s) == 0
