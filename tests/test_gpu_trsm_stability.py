"""Backward error of the triangular solves where a 16 x 16 diagonal block is far worse
conditioned than its entries show: such a block has to be substituted, its explicit inverse
would lose the digits (a factor of 1e5 and more in the residual below).

Measure: max |op(T) X - alpha B| / (|op(T)| |X| + |alpha B|), element by element, the residual in
long double.  Substitution of an order n keeps it below n * u to first order whatever the
condition of T, as do the products between the blocks (Higham, Accuracy and Stability, theorems
8.5 and 3.5; u = eps / 2); a block that is inverted all the same may add 16 u.  Tolerance:
(n + 16) * u.
"""
import math

import numpy as np
import pytest

from _devmem import Matrix

pytestmark = pytest.mark.gpu
U = np.finfo(np.float64).eps / 2
FORMS = [("L", "N"), ("L", "T"), ("U", "N"), ("U", "T")]


def _solve_order(rng, n, unit):
    """A lower triangle, rows in the order in which they are solved: the first, a middle and the
    last diagonal block of 16 ill conditioned (off-diagonal entries up to 4 beside ones), the
    others as a factorisation leaves them."""
    t = np.tril(rng.uniform(-1, 1, (n, n)), -1) / (math.sqrt(n) if unit else 1)
    t[np.arange(n), np.arange(n)] = 1 if unit else math.sqrt(n) * (1 + rng.uniform(0, 1, n))
    for b in {0, (n // 32) * 16, (n - 1) // 16 * 16}:
        r = slice(b, min(n, b + 16))
        k = r.stop - b
        t[r, r] = np.tril(rng.uniform(-4, 4, (k, k)), -1) + np.eye(k)
    return t


def _stored(t, uplo, trans):
    """The matrix whose op() is t read forwards (a lower op) or backwards (an upper one)."""
    if (uplo == "L") == (trans == "N"):
        m = t
    else:
        m = t[::-1, ::-1]
    return np.asfortranarray(m if trans == "N" else m.T)


def _error(a, uplo, trans, unit, x, b):
    t = (np.tril(a) if uplo == "L" else np.triu(a)).astype(np.longdouble)
    if unit:
        np.fill_diagonal(t, 1)
    t = t if trans == "N" else t.T
    x, b = x.astype(np.longdouble), b.astype(np.longdouble)
    return float(np.max(np.abs(t @ x - b) / (np.abs(t) @ np.abs(x) + np.abs(b))))


def _system(n, nrhs, uplo, trans, unit):
    rng = np.random.default_rng(n)
    a = _stored(_solve_order(rng, n, unit), uplo, trans)
    t = (np.tril(a) if uplo == "L" else np.triu(a)).astype(np.longdouble)
    t = t if trans == "N" else t.T
    b = (t @ rng.uniform(-1, 1, (n, nrhs))).astype(np.float64)
    if unit:
        np.fill_diagonal(a, 7.0)  # never read
    return a, b


@pytest.mark.parametrize("unit", [False, True])
@pytest.mark.parametrize("side", "LR")
@pytest.mark.parametrize("uplo,trans", FORMS)
def test_call(gpu, side, uplo, trans, unit):
    # X op(A) = B is op(A)^T X^T = B^T
    t = trans if side == "L" else ("T" if trans == "N" else "N")
    for n in (16, 23, 128, 200, 256, 300, 512, 600):
        a, b = _system(n, 18, uplo, t, unit)
        x = np.array(b if side == "L" else b.T, order="F")
        gpu.dtrsm(side, uplo, trans, "U" if unit else "N", x.shape[0], x.shape[1], 1.0, a, n, x,
                  x.shape[0])
        err = _error(a, uplo, t, unit, x if side == "L" else x.T, b)
        assert err <= (n + 16) * U, (n, err / U)


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("uplo,trans", FORMS)
def test_batch(gpu, uplo, trans, graph):
    slot = gpu.Batch(use_graph=graph)
    try:
        for n in (16, 23, 256, 300, 512, 700, 1024):
            a, b = _system(n, 18, uplo, trans, False)
            A, B = Matrix(gpu, a), Matrix(gpu, b)
            assert slot.dtrsm("L", uplo, trans, "N", n, 18, 1.0, A.ptr, n, B.ptr, n) == 0
            slot.run()
            err = _error(a, uplo, trans, False, B.get(), b)
            A.free()
            B.free()
            assert err <= (n + 16) * U, (n, err / U)
    finally:
        slot.close()


@pytest.mark.parametrize("trans", "NT")
@pytest.mark.parametrize("batch", [False, True])
def test_least_squares_factor(gpu, trans, batch):
    """R of the QR factorisation of a 64-point monomial basis of 16 terms."""
    r = np.asfortranarray(np.linalg.qr(np.vander(np.linspace(0, 1, 64), 16, increasing=True))[1])
    op = r.astype(np.longdouble) if trans == "N" else r.astype(np.longdouble).T
    b = np.asfortranarray((op @ np.random.default_rng(1).uniform(-1, 1, (16, 20))).astype(np.float64))
    if batch:
        R, X, slot = Matrix(gpu, r), Matrix(gpu, b), gpu.Batch(use_graph=False)
        try:
            assert slot.dtrsm("L", "U", trans, "N", 16, 20, 1.0, R.ptr, 16, X.ptr, 16) == 0
            slot.run()
            x = X.get()
        finally:
            slot.close()
            R.free()
            X.free()
    else:
        x = b.copy(order="F")
        gpu.dtrsm("L", "U", trans, "N", 16, 20, 1.0, r, 16, x, 16)
    assert _error(r, "U", trans, False, x, b) <= 32 * U


@pytest.mark.parametrize("uplo,trans", FORMS)
def test_inverse_overflows(gpu, uplo, trans):
    """Finite triangles whose inverse is not: diagonal 1e-160, off-diagonal entries to 1e150."""
    for n in (5, 16, 40, 300):
        rng = np.random.default_rng(n)
        t = np.tril(rng.uniform(-1e150, 1e150, (n, n)), -1)
        t[np.arange(n), np.arange(n)] = 1e-160 * (1 + rng.uniform(0, 1, n))
        a = _stored(t, uplo, trans)
        # rows that are solved first give zeros, the last one its quotient
        last = -1 if (uplo == "L") == (trans == "N") else 0
        b = np.zeros((n, 3), order="F")
        b[last] = (1e-160, -2e-160, 3e100)
        want = np.zeros((n, 3))
        want[last] = b[last] / a[last, last]
        gpu.dtrsm("L", uplo, trans, "N", n, 3, 1.0, a, n, b, n)
        assert np.all(np.abs(b - want) <= 4 * U * np.abs(want)), n


@pytest.mark.parametrize("uplo,trans", FORMS)
def test_single(gpu, uplo, trans):
    """FP32 orders up to 512 are solved in FP64: a rounding of the result is all that is left."""
    for n in (16, 128, 256, 300, 512):
        a, b = (v.astype(np.float32) for v in _system(n, 18, uplo, trans, False))
        x = np.array(b, order="F")
        gpu.strsm("L", uplo, trans, "N", n, 18, 1.0, np.asfortranarray(a), n, x, n)
        assert _error(a, uplo, trans, False, x, b) <= np.finfo(np.float32).eps, n


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("uplo,trans", FORMS)
def test_limits_of_the_type(gpu, uplo, trans, batch):
    """A NaN in one right-hand side, in the next a diagonal entry whose reciprocal is infinite
    (and not the quotient), in the others a sum of products that is infinite (and not what remains
    of B when they are subtracted one by one: two roundings, u * 1.8e308 at most)."""
    for n in (7, 17, 40, 128, 200, 256, 300, 512):
        mid = n // 2 | 1
        t, b = np.eye(n), np.zeros((n, 18))
        t[n - 1, [0, mid]] = 0.9
        t[n - 2, n - 2] = 1e-310
        b[0, 0] = np.nan
        b[n - 2, 1] = 1e-310
        b[[0, mid, n - 1], 2:] = 1e308
        want = b.copy()
        want[n - 2, 1] = 1
        want[n - 1, 2:] = -0.8e308
        a = _stored(t, uplo, trans)
        step = 1 if (uplo == "L") == (trans == "N") else -1
        x = np.array(b[::step], order="F")
        if batch:
            A, X, slot = Matrix(gpu, a), Matrix(gpu, x), gpu.Batch(use_graph=False)
            try:
                assert slot.dtrsm("L", uplo, trans, "N", n, 18, 1.0, A.ptr, n, X.ptr, n) == 0
                slot.run()
                x = X.get()
            finally:
                slot.close()
                A.free()
                X.free()
        else:
            gpu.dtrsm("L", uplo, trans, "N", n, 18, 1.0, a, n, x, n)
        x = x[::step]
        assert np.isnan(x[0, 0]), n
        assert np.array_equal(x[: n - 1, 1:], want[: n - 1, 1:]) and x[n - 1, 1] == 0, n
        assert np.abs(x[n - 1, 2:] + 0.8e308).max() <= U * 1.8e308, n
