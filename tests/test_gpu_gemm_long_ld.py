"""Products whose leading dimensions lie at the limit of the fast tile's 32-bit lane offsets (2^24)
and past it, where the 64-bit forms run: plain, split along k, and on a triangular grid, operands
read along and across their columns.  Small integers: every sum is exact.  Only the rows that a
product reads are written; the rest of the (up to 10 GB) operand is whatever the memory held."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
VP, CI, SZ = ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t
LIMIT = 1 << 24


class Long:
    """The rows of `a` at the head of columns `ld` apart, on the device."""

    def __init__(self, lib, a, ld):
        self.lib, self.a, self.ld = lib, np.asfortranarray(a), ld
        rows, cols = a.shape
        self.ptr = lib.gpublas_dev_alloc(SZ(((cols - 1) * ld + rows) * a.itemsize))
        if not self.ptr:
            pytest.skip("no device memory for the operand")
        assert lib.gpublas_dev_h2d_2d(VP(self.ptr), SZ(ld), VP(self.a.ctypes.data), SZ(rows), SZ(rows),
                                      SZ(cols), SZ(a.itemsize), None) == 0
        assert lib.gpublas_dev_sync(None) == 0

    def get(self):
        out = np.empty_like(self.a)
        rows, cols = out.shape
        assert self.lib.gpublas_dev_d2h_2d(VP(out.ctypes.data), SZ(rows), VP(self.ptr), SZ(self.ld),
                                           SZ(rows), SZ(cols), SZ(out.itemsize), None) == 0
        assert self.lib.gpublas_dev_sync(None) == 0
        return out

    def free(self):
        self.lib.gpublas_dev_release(VP(self.ptr))


@pytest.mark.parametrize("prec", "ds")
@pytest.mark.parametrize("ld", [LIMIT, LIMIT + 1])
@pytest.mark.parametrize("ta,tb,m,n,k", [
    ("T", "N", 70, 67, 100),   # both along k
    ("T", "N", 64, 33, 600),   # the same, split along k
    ("N", "T", 70, 65, 41),    # both across k
    ("N", "N", 100, 64, 37),
    ("T", "T", 40, 70, 50),    # narrower than 64: generic past the limit
])
def test_product(gpu, prec, ld, ta, tb, m, n, k):
    lib = gpu.library()
    f, real, dt = ((lib.gpublas_dev_dgemm, ctypes.c_double, np.float64) if prec == "d" else
                   (lib.gpublas_dev_sgemm, ctypes.c_float, np.float32))
    rng = np.random.default_rng(m + k)
    a, b, c = (rng.integers(-3, 4, s).astype(dt) for s in ((m, k), (k, n), (m, n)))
    A = Long(lib, a if ta == "N" else a.T, ld)
    B = Long(lib, b if tb == "N" else b.T, b.shape[0 if tb == "N" else 1])
    C = Long(lib, c, m)
    try:
        for x, y, side in ((A, B, "left"), (B, A, "right")):
            # the long operand on the left, then (transposed product) on the right
            if side == "left":
                err = f(None, ctypes.c_char(ta.encode()), ctypes.c_char(tb.encode()), CI(m), CI(n),
                        CI(k), real(1.0), VP(x.ptr), CI(x.ld), VP(y.ptr), CI(y.ld), real(2.0),
                        VP(C.ptr), CI(m))
                want = a @ b + 2 * c
            else:
                C.free()
                C = Long(lib, c.T.copy(), n)
                flip = {"N": b"T", "T": b"N"}
                err = f(None, ctypes.c_char(flip[tb]), ctypes.c_char(flip[ta]), CI(n), CI(m), CI(k),
                        real(1.0), VP(x.ptr), CI(x.ld), VP(y.ptr), CI(y.ld), real(2.0), VP(C.ptr),
                        CI(n))
                want = (a @ b + 2 * c).T
            assert err == 0 and np.array_equal(C.get(), want), side
    finally:
        for x in (A, B, C):
            x.free()
        lib.gpublas_dev_trim()


@pytest.mark.parametrize("prec", "ds")
@pytest.mark.parametrize("trans,n,k", [("T", 70, 90), ("N", 90, 40)])
def test_rank_k(gpu, prec, trans, n, k):
    lib = gpu.library()
    f, real, dt = ((lib.gpublas_dev_dsyrk, ctypes.c_double, np.float64) if prec == "d" else
                   (lib.gpublas_dev_ssyrk, ctypes.c_float, np.float32))
    rng = np.random.default_rng(n)
    a = rng.integers(-3, 4, (n, k)).astype(dt)
    c = rng.integers(-3, 4, (n, n)).astype(dt)
    A, C = Long(lib, a if trans == "N" else a.T, LIMIT + 1), Long(lib, c, n)
    try:
        assert f(None, ctypes.c_char(b"L"), ctypes.c_char(trans.encode()), CI(n), CI(k), real(1.0),
                 VP(A.ptr), CI(LIMIT + 1), real(1.0), VP(C.ptr), CI(n)) == 0
        low = np.tril(np.ones((n, n), bool))
        assert np.array_equal(C.get(), np.where(low, a @ a.T + c, c))
    finally:
        A.free()
        C.free()
        lib.gpublas_dev_trim()
