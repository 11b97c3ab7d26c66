"""The 16-column triangular panel solve at the orders where its blocks, its waves
and its variants change, in every side / uplo / trans / diag form, per call and in
a batch slot, and its substitution for results that are not finite.

Reference: substitution in numpy's 80-bit long double.  The triangles are those of
a factorisation (off-diagonal entries in [-1, 1], diagonal sqrt(n) (1 + u)), whose
condition is of order one, so the solve's own bound n * eps (Higham, Accuracy and
Stability, 8.5) is the tolerance; in FP32 an order of at most 512 is solved in FP64
and rounded once: eps / 2 per element.
"""
import math

import numpy as np
import pytest

from _devmem import Matrix

pytestmark = pytest.mark.gpu
EPS64, EPS32 = np.finfo(np.float64).eps, np.finfo(np.float32).eps
FORMS = [(s, u, t, d) for s in "LR" for u in "LU" for t in "NT" for d in "NU"]


def _triangle(rng, n, diag, dt):
    a = rng.uniform(-1, 1, (n, n))
    if diag == "U":
        a /= math.sqrt(n)  # the stored diagonal is not read
    else:
        a[np.arange(n), np.arange(n)] = math.sqrt(n) * (1 + rng.uniform(0, 1, n))
    return a.astype(dt)


def _substitute(a, b, uplo, trans, diag):
    """op(A) X = B in long double, A's other triangle not read."""
    n = a.shape[0]
    t = (np.tril(a) if uplo == "L" else np.triu(a)).astype(np.longdouble)
    if diag == "U":
        np.fill_diagonal(t, 1)
    t = t if trans == "N" else t.T
    x = b.astype(np.longdouble)
    forward = (uplo == "L") == (trans == "N")
    for k in range(n) if forward else range(n - 1, -1, -1):
        x[k] /= t[k, k]
        rest = slice(k + 1, n) if forward else slice(0, k)
        x[rest] -= t[rest, k:k + 1] * x[k]
    return x


def _place(gb, a, ld, off):
    """`a` in a tracked matrix of leading dimension ld that starts at element `off`."""
    flat = gb.tracked_empty((off + ld * a.shape[1],), a.dtype)
    flat[:] = 7.0
    m = flat[off:].reshape((ld, a.shape[1]), order="F")
    m[:a.shape[0]] = a
    return m


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("side,uplo,trans,diag", FORMS)
def test_panel_orders(gpu, single, side, uplo, trans, diag):
    dt, eps = (np.float32, EPS32) if single else (np.float64, EPS64)
    f = gpu.strsm if single else gpu.dtrsm
    for n, nrhs in ((1, 1), (15, 17), (16, 16), (17, 15), (113, 3), (128, 33), (129, 16), (241, 5),
                    (256, 17), (257, 16), (300, 20), (497, 1), (512, 31), (513, 18), (700, 16)):
        rng = np.random.default_rng(n)
        a, x0 = _triangle(rng, n, diag, dt), rng.uniform(-1, 1, (n, nrhs)).astype(dt)
        b = x0 if side == "L" else np.ascontiguousarray(x0.T)
        A, B = _place(gpu, a, n + 1, 1), _place(gpu, b, b.shape[0] + 1, 1)
        f(side, uplo, trans, diag, b.shape[0], b.shape[1], 1.0, A, n + 1, B, b.shape[0] + 1)
        got = np.array(B)
        assert np.all(got[b.shape[0]:] == 7.0)
        got = got[:b.shape[0]] if side == "L" else got[:b.shape[0]].T
        # X op(A) = B is op(A)^T X^T = B^T
        t = trans if side == "L" else ("T" if trans == "N" else "N")
        want = _substitute(a, x0, uplo, t, diag)
        err = np.linalg.norm((got - want).astype(np.float64)) / np.linalg.norm(want.astype(np.float64))
        assert err <= (eps if single and n <= 512 else n * eps), (n, nrhs, err)


@pytest.mark.parametrize("uplo,trans", [("L", "N"), ("L", "T"), ("U", "N"), ("U", "T")])
@pytest.mark.parametrize("diag", ["N", "U"])
def test_batch_panel_orders(gpu, uplo, trans, diag):
    for m, n in ((1, 16), (33, 5), (256, 17), (257, 16), (512, 20), (513, 16), (900, 3), (1024, 18)):
        rng = np.random.default_rng(m)
        a, b = _triangle(rng, m, diag, np.float64), rng.uniform(-1, 1, (m, n))
        A, B = Matrix(gpu, a), Matrix(gpu, b)
        slot = gpu.Batch(use_graph=False)
        try:
            assert slot.dtrsm("L", uplo, trans, diag, m, n, 2.0, A.ptr, m, B.ptr, m) == 0
            slot.run()
        finally:
            slot.close()
        got, want = B.get(), _substitute(a, 2.0 * b, uplo, trans, diag)
        err = np.linalg.norm((got - want).astype(np.float64)) / np.linalg.norm(want.astype(np.float64))
        A.free()
        B.free()
        assert err <= m * EPS64, (m, n, err)


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("uplo,trans", [("L", "N"), ("U", "N"), ("L", "T")])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_panel_rows_before_a_non_finite_one(gpu, single, uplo, trans, bad):
    """An infinity or NaN in one right-hand side reaches the rows solved after it in that column
    and nothing else; a zero on the diagonal the rows from it on."""
    dt, eps = (np.float32, EPS32) if single else (np.float64, EPS64)
    f = gpu.strsm if single else gpu.dtrsm
    forward = (uplo == "L") == (trans == "N")
    for n, at in ((40, 21), (200, 100), (300, 290)):
        rng = np.random.default_rng(n)
        a, b = _triangle(rng, n, "N", dt), np.asfortranarray(rng.uniform(-1, 1, (n, 20)).astype(dt))
        want = _substitute(a, b, uplo, trans, "N").astype(np.float64)
        before = slice(0, at) if forward else slice(at + 1, n)
        b[at, 3] = bad
        A = np.asfortranarray(a)
        x = b.copy(order="F")
        f("L", uplo, trans, "N", n, 20, 1.0, A, n, x, n)
        clean = [c for c in range(20) if c != 3]
        tol = n * eps * np.abs(want).max()
        assert np.abs(x[:, clean] - want[:, clean]).max() <= tol
        assert np.abs(x[before, 3] - want[before, 3]).max() <= tol
        assert not np.isfinite(x[at, 3])
        A[at, at] = 0.0
        x = np.asfortranarray(np.where(np.isfinite(b), b, 1).astype(dt))
        f("L", uplo, trans, "N", n, 20, 1.0, A, n, x, n)
        assert np.abs(x[before][:, clean] - want[before][:, clean]).max() <= tol
        assert not np.isfinite(x[at]).any()
