"""Level-2 kernels on columns that start at any element: odd leading dimensions, operands one
element into their allocation, odd row counts (the 16-byte accesses then straddle lines, and the
last row goes alone).  Small integers: sums are exact, results compared bit for bit with numpy;
rows past m must come back untouched.  The solves use a triangle of order-one condition and the
bound n * eps against long double."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps
SHAPES = [(1, 1), (2, 3), (127, 130), (511, 9), (513, 17), (515, 40), (1025, 1031)]


def _put(gb, a, pad, off=1):
    ld = a.shape[0] + pad
    flat = gb.tracked_empty((off + ld * a.shape[1],))
    flat[:] = -5.0
    m = flat[off:].reshape((ld, a.shape[1]), order="F")
    m[:a.shape[0]] = a
    return m, ld


def _vec(gb, v, inc=1):
    flat = gb.tracked_empty((1 + (len(v) - 1) * abs(inc) + 1,))
    flat[:] = -7.0
    x = flat[1:]
    x[::abs(inc)][:len(v)] = v if inc > 0 else v[::-1]
    return x


def _ints(rng, *shape):
    return rng.integers(-3, 4, shape).astype(np.float64)


@pytest.mark.parametrize("pad", [0, 1, 2])
@pytest.mark.parametrize("m,n", SHAPES)
def test_gemv_ger(gpu, m, n, pad):
    rng = np.random.default_rng(m + pad)
    a, u, v = _ints(rng, m, n), _ints(rng, m), _ints(rng, n)
    A, ld = _put(gpu, a, pad)
    for trans, x, y0, want in (("N", v, u, 2 * (a @ v) - u), ("T", u, v, 2 * (a.T @ u) - v)):
        for incx in (1, -2):
            X, Y = _vec(gpu, x, incx), _vec(gpu, y0)
            gpu.dgemv(trans, m, n, 2.0, A, ld, X, incx, -1.0, Y, 1)
            assert np.array_equal(np.array(Y)[:len(want)], want)
    gpu.dger(m, n, 3.0, _vec(gpu, u), 1, _vec(gpu, v), 1, A, ld)
    got = np.array(A)
    assert np.array_equal(got[:m], a + 3 * np.outer(u, v))
    assert np.all(got[m:] == -5.0)


@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("n", [1, 2, 127, 128, 129, 255, 257, 515])
def test_symmetric_and_triangular(gpu, uplo, n):
    rng = np.random.default_rng(n)
    a, x, y = _ints(rng, n, n), _ints(rng, n), _ints(rng, n)
    tri = np.tril(a) if uplo == "L" else np.triu(a)
    full = tri + tri.T - np.diag(np.diag(a))
    A, ld = _put(gpu, a, 1 - n % 2)  # odd leading dimension
    Y = _vec(gpu, y)
    gpu.dsymv(uplo, n, 2.0, A, ld, _vec(gpu, x), 1, 3.0, Y, 1)
    assert np.array_equal(np.array(Y)[:n], 2 * (full @ x) + 3 * y)
    for trans, want in (("N", tri @ x), ("T", tri.T @ x)):
        X = _vec(gpu, x)
        gpu.dtrmv(uplo, trans, "N", n, A, ld, X, 1)
        assert np.array_equal(np.array(X)[:n], want)
    keep = np.tri(n, dtype=bool) if uplo == "L" else np.tri(n, dtype=bool).T
    gpu.dsyr(uplo, n, 2.0, _vec(gpu, x), 1, A, ld)
    want = np.where(keep, a + 2 * np.outer(x, x), a)
    assert np.array_equal(np.array(A)[:n], want)
    gpu.dsyr2(uplo, n, -1.0, _vec(gpu, x), 1, _vec(gpu, y), 1, A, ld)
    assert np.array_equal(np.array(A)[:n], np.where(keep, want - np.outer(x, y) - np.outer(y, x), a))


@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("n", [1, 33, 127, 129, 385, 700])
def test_solves(gpu, uplo, trans, n):
    rng = np.random.default_rng(n)
    a = rng.uniform(-1, 1, (n, n))
    a[np.arange(n), np.arange(n)] = math.sqrt(n) * (1 + rng.uniform(0, 1, n))
    b = rng.uniform(-1, 1, n)
    t = (np.tril(a) if uplo == "L" else np.triu(a)).astype(np.longdouble)
    t = t if trans == "N" else t.T
    want = b.astype(np.longdouble)
    forward = (uplo == "L") == (trans == "N")
    for k in range(n) if forward else range(n - 1, -1, -1):
        want[k] /= t[k, k]
        rest = slice(k + 1, n) if forward else slice(0, k)
        want[rest] -= t[rest, k] * want[k]
    A, ld = _put(gpu, a, 1 - n % 2)
    packed = np.concatenate([a[j:, j] if uplo == "L" else a[:j + 1, j] for j in range(n)])
    P, X, Z = _vec(gpu, packed), _vec(gpu, b), _vec(gpu, b)
    gpu.dtrsv(uplo, trans, "N", n, A, ld, X, 1)
    gpu.dtpsv(uplo, trans, "N", n, P, Z, 1)
    for got in (X, Z):
        err = np.linalg.norm((np.array(got)[:n] - want).astype(np.float64))
        assert err <= n * EPS * np.linalg.norm(want.astype(np.float64))
