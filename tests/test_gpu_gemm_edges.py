"""The fast GEMM tile where it can go wrong: ragged rows and columns (the last
tile moved back over its neighbour), every remainder of the k pipeline, operands
that start at an odd element, odd leading dimensions, ragged triangular grids and
ragged triangular-k products.

Integer data whose sums stay below 2^24: every correct result is bit-exact, and
numpy's product of the same integers in float64 is the reference.  Rows past m
in every column, and the other triangle, must come back untouched.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROGUE = -77.0


def _matrix(gb, rng, rows, cols, ld, off, dt):
    """A tracked ld x cols matrix that starts `off` elements into its object."""
    flat = gb.tracked_empty((off + ld * cols,), dt)
    host = np.full(off + ld * cols, ROGUE, dt)
    view = host[off:].reshape((ld, cols), order="F")
    view[:rows, :] = rng.integers(-3, 4, size=(rows, cols))
    flat[:] = host
    return flat[off:].reshape((ld, cols), order="F"), view


def _gemm(gb, single, ta, tb, m, n, k, pad, off, beta):
    dt = np.float32 if single else np.float64
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    ra, ca = (m, k) if ta == "N" else (k, m)
    rb, cb = (k, n) if tb == "N" else (n, k)
    A, ha = _matrix(gb, rng, ra, ca, ra + pad, off, dt)
    B, hb = _matrix(gb, rng, rb, cb, rb + pad, off, dt)
    C, hc = _matrix(gb, rng, m, n, m + pad, off, dt)
    f = gb.sgemm if single else gb.dgemm
    f(ta, tb, m, n, k, 2.0, A, ra + pad, B, rb + pad, beta, C, m + pad)
    a, b = ha[:ra].astype(np.float64), hb[:rb].astype(np.float64)
    want = 2.0 * ((a if ta == "N" else a.T) @ (b if tb == "N" else b.T)) + beta * hc[:m]
    got = np.array(C)
    assert np.array_equal(got[:m], want)
    assert np.array_equal(got[m:], hc[m:])


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("m,n,k", [
    (32, 32, 1), (33, 47, 16), (40, 34, 33), (31, 64, 40), (45, 70, 1000), (32, 33, 5000),
    (64, 64, 1), (64, 65, 15), (65, 64, 16), (127, 66, 17), (128, 129, 31), (129, 127, 32),
    (191, 193, 33), (64, 200, 47), (63, 65, 48), (200, 63, 49), (65, 66, 1000)])
def test_gemm_tile_edges(gpu, single, ta, tb, m, n, k):
    """32 x 32 and 64 x 64 tiles (the generic tile below 32), k from one step to a split k."""
    _gemm(gpu, single, ta, tb, m, n, k, pad=1, off=1, beta=-1.0)
    _gemm(gpu, single, ta, tb, m, n, k, pad=0, off=0, beta=0.0)


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("m,n,k", [(2049, 2055, 33), (2944, 2816, 48), (129, 32769, 18),
                                   (1030, 1100, 130), (2816, 2910, 161)])
def test_gemm_large_tile_edges(gpu, single, ta, tb, m, n, k):
    """Products large enough for 64 x 64 tiles at every stage of the k pipeline, and for
    128 x 64 (FP64) and 128 x 128 (FP32) ones, ragged in both dimensions."""
    _gemm(gpu, single, ta, tb, m, n, k, pad=3, off=1, beta=1.0)


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("n,k", [(64, 5), (65, 16), (190, 33), (2050, 40), (4100, 17)])
def test_syrk_ragged_triangle(gpu, single, uplo, trans, n, k):
    """Triangular grids with a ragged last tile row: the tile moved back overlaps
    its neighbours and the diagonal, and writes neither."""
    dt = np.float32 if single else np.float64
    rng = np.random.default_rng(n + k)
    ra, ca = (n, k) if trans == "N" else (k, n)
    A, ha = _matrix(gpu, rng, ra, ca, ra + 1, 1, dt)
    C, hc = _matrix(gpu, rng, n, n, n + 1, 1, dt)
    f = gpu.ssyrk if single else gpu.dsyrk
    f(uplo, trans, n, k, 1.0, A, ra + 1, -2.0, C, n + 1)
    a = ha[:ra].astype(np.float64)
    want = hc.astype(np.float64)
    full = (a @ a.T if trans == "N" else a.T @ a) - 2.0 * want[:n]
    keep = np.tri(n, dtype=bool) if uplo == "L" else np.tri(n, dtype=bool).T
    want[:n][keep] = full[keep]
    assert np.array_equal(np.array(C), want)


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("side", ["L", "R"])
@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("m,n", [(65, 130), (201, 67), (2050, 2100)])
def test_trmm_ragged_range(gpu, single, side, uplo, trans, m, n):
    """Products over the nonzero k range of a triangle, ragged in both dimensions."""
    dt = np.float32 if single else np.float64
    rng = np.random.default_rng(m + n)
    na = m if side == "L" else n
    A, ha = _matrix(gpu, rng, na, na, na + 1, 1, dt)
    B, hb = _matrix(gpu, rng, m, n, m + 1, 1, dt)
    f = gpu.strmm if single else gpu.dtrmm
    f(side, uplo, trans, "N", m, n, 2.0, A, na + 1, B, m + 1)
    t = np.tril(ha[:na]) if uplo == "L" else np.triu(ha[:na])
    t = (t if trans == "N" else t.T).astype(np.float64)
    want = hb.astype(np.float64)
    want[:m] = 2.0 * (t @ want[:m] if side == "L" else want[:m] @ t)
    assert np.array_equal(np.array(B), want)


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("m,n,k", [(500, 449, 16411), (129, 2000, 10007)])
def test_long_k_split_on_64(gpu, ta, tb, m, n, k):
    """FP32 products past 128 tiles of 32 x 32 whose k is long enough to split on 64 x 64 ones,
    the last tiles and the last chunk ragged.  Sums stay below 2^24, so they are exact."""
    rng = np.random.default_rng(k)
    a, b = (rng.integers(-3, 4, s).astype(np.float32) for s in ((m, k), (k, n)))
    want = a.astype(np.float64) @ b.astype(np.float64)
    A, B = (np.asfortranarray(x if t == "N" else x.T) for x, t in ((a, ta), (b, tb)))
    C = np.full((m, n), 3.0, np.float32, order="F")
    gpu.sgemm(ta, tb, m, n, k, 1.0, A, A.shape[0], B, B.shape[0], -1.0, C, m)
    assert np.array_equal(C, want - 3.0)
