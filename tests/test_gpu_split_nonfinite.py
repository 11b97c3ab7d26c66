"""Split products with an Inf or NaN among the inputs: the product kernels leave C alone and the
FP64 kernel computes it, in every slice format, rectangular and triangular, at ragged sizes and
at line lengths around the eight-element steps of the exponent passes.  Bit for bit the plain
FP64 product of the same call."""
import ctypes

import numpy as np
import pytest

from _devmem import Matrix

pytestmark = pytest.mark.gpu
FORMATS = [(0, 6), (1, 5), (2, 7)]  # BF16, FP16, INT8 with their slices


def _call(gpu, f, *args):
    conv = [ctypes.c_char(a.encode()) if isinstance(a, str) else ctypes.c_double(a)
            if isinstance(a, float) else ctypes.c_void_p(a.ptr) if isinstance(a, Matrix)
            else a for a in args]
    assert f(None, *conv) == 0
    gpu.sync()


@pytest.mark.parametrize("fmt,slices", FORMATS)
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("m,n,k,at", [(70, 65, 33, (0, 0)), (130, 64, 71, (129, 70)),
                                      (64, 200, 600, (13, 517))])
def test_gemm(gpu, fmt, slices, bad, m, n, k, at):
    lib = gpu.library()
    rng = np.random.default_rng(m)
    a, b, c = (rng.uniform(-1, 1, s) for s in ((m, k), (k, n), (m, n)))
    for inject in (None, "a", "b"):
        if inject:
            (a if inject == "a" else b.T)[at[0] % (m if inject == "a" else n), at[1]] = bad
        for ta, tb in (("N", "N"), ("T", "T")):
            A = Matrix(gpu, a if ta == "N" else a.T)
            B = Matrix(gpu, b if tb == "N" else b.T)
            C, D = Matrix(gpu, c), Matrix(gpu, c)
            shape = (ta, tb, m, n, k, 1.5, A, A.like.shape[0], B, B.like.shape[0], -0.5)
            _call(gpu, lib.gpublas_dev_dgemm_split_fmt, slices, fmt, *shape, C, m)
            _call(gpu, lib.gpublas_dev_dgemm, *shape, D, m)
            got, plain = C.get(), D.get()
            for x in (A, B, C, D):
                x.free()
            if inject:
                assert np.array_equal(got, plain, equal_nan=True)
            else:
                # s slices of w bits leave k products of relative size 2^-(w s) each
                w = 7 if fmt == 2 else 8
                bound = 4 * k * 2.0 ** -(w * slices) + 64 * np.finfo(float).eps * np.sqrt(k)
                assert np.abs(got - plain).max() <= bound * 1.5
        if inject == "a":
            a = rng.uniform(-1, 1, (m, k))


@pytest.mark.parametrize("fmt,slices", FORMATS)
@pytest.mark.parametrize("uplo,trans", [("L", "N"), ("U", "T")])
def test_syrk(gpu, fmt, slices, uplo, trans):
    lib = gpu.library()
    n, k = 133, 75
    rng = np.random.default_rng(3)
    a, c = rng.uniform(-1, 1, (n, k)), rng.uniform(-1, 1, (n, n))
    a[100, 40] = np.nan
    A = Matrix(gpu, a if trans == "N" else a.T)
    C, D = Matrix(gpu, c), Matrix(gpu, c)
    shape = (uplo, trans, n, k, 1.0, A, A.like.shape[0], 0.25)
    _call(gpu, lib.gpublas_dev_dsyrk_split_fmt, slices, fmt, *shape, C, n)
    _call(gpu, lib.gpublas_dev_dsyrk, *shape, D, n)
    assert np.array_equal(C.get(), D.get(), equal_nan=True)
    for x in (A, C, D):
        x.free()
