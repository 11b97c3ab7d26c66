"""DTRMM with as many large tiles as its 128 x 64 form takes, the triangle's order a few ragged
tiles, in every side / uplo / trans form.  Small integers: every sum is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", "LR")
@pytest.mark.parametrize("uplo", "LU")
@pytest.mark.parametrize("trans", "NT")
def test_dtrmm_large_tiles(gpu, side, uplo, trans):
    na, nb = 200, 200003
    m, n = (na, nb) if side == "L" else (nb, na)
    rng = np.random.default_rng(5)
    a = np.asfortranarray(rng.integers(-2, 3, (na, na)).astype(float))
    b = np.asfortranarray(rng.integers(-2, 3, (m, n), dtype=np.int8).astype(float))
    t = np.tril(a) if uplo == "L" else np.triu(a)
    t = t if trans == "N" else t.T
    want = t @ b if side == "L" else b @ t
    gpu.dtrmm(side, uplo, trans, "N", m, n, 1.0, a, na, b, m)
    assert np.array_equal(b, want)
