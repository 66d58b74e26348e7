"""Cholesky, panel and triangular-inverse kernels at the orders where their
tiles end (16), their leaves end (128), a block column ends (512) and the
schedule changes (1024), with the bars of the reference's drivers: ||A - L
L^T|| / (N ||A|| eps) <= 10 and ||A X - B|| / ((||A|| ||X|| + ||B||) N eps) <=
10.  The triangle that is not referenced holds NaN and keeps it."""
import numpy as np
import pytest

from helpers import rng, spd, tri_matrix, uniform

pytestmark = pytest.mark.gpu

ORDERS = [1, 2, 15, 16, 17, 63, 64, 65, 112, 113, 127, 128, 129, 144, 255, 257, 385, 511, 513, 640, 1023, 1025, 1537]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("uplo", [121, 122])
@pytest.mark.parametrize("n", ORDERS)
def test_potrf_block_edges(xk, n, uplo, dtype):
    r = rng(n + uplo)
    A = spd(r, n, dtype)
    off = np.triu_indices(n, 1) if uplo == 122 else np.tril_indices(n, -1)
    F = A.copy(order="F")
    F[off] = np.nan
    assert xk.potrf(uplo, F) == 0
    xk.invalidate()
    assert np.all(np.isnan(F[off]))
    F[off] = 0
    L = (F if uplo == 122 else F.T).astype(np.float64)
    A = A.astype(np.float64)
    res = np.abs(A - L @ L.T).sum(axis=1).max() / (n * np.abs(A).sum(axis=1).max() * np.finfo(dtype).eps)
    assert res <= 10, res


@pytest.mark.parametrize("uplo", [121, 122])
@pytest.mark.parametrize("n,bad", [(16, 0), (16, 15), (40, 16), (128, 127), (200, 130), (600, 511), (600, 512),
                                   (1300, 1100)])
def test_potrf_failing_order(xk, n, bad, uplo):
    A = spd(rng(n), n)
    A[bad, bad] = -1.0
    assert xk.potrf(uplo, A) == bad + 1
    xk.invalidate()


@pytest.mark.parametrize("uplo", [121, 122])
def test_potrf_diagonal_of_any_exponent(xk, uplo):
    """The pivots' reciprocals neither overflow nor lose a denormal."""
    n = 150
    d = 2.0 ** rng(5).integers(-1060, 1020, n)
    F = np.asfortranarray(np.diag(d))
    assert xk.potrf(uplo, F) == 0
    xk.invalidate()
    assert np.allclose(np.diag(F), np.sqrt(d), rtol=4 * np.finfo(np.float64).eps, atol=0)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("diag", [131, 132])
@pytest.mark.parametrize("uplo", [121, 122])
@pytest.mark.parametrize("n", [1, 16, 17, 64, 65, 127, 128, 129, 300, 384, 513, 1100])
def test_trsm_block_edges(xk, n, uplo, diag, dtype):
    r = rng(n + uplo + diag)
    A = tri_matrix(r, n, uplo == 122, diag == 132, dtype)
    if diag == 131:
        A[np.diag_indices(n)] = r.uniform(1.0, 2.0, n)
    T = (np.tril(A) if uplo == 122 else np.triu(A)).astype(np.float64)
    A[np.triu_indices(n, 1) if uplo == 122 else np.tril_indices(n, -1)] = np.nan
    if diag == 132:
        A[np.diag_indices(n)] = np.nan
    B = uniform(r, n, 19, dtype=dtype)
    X = B.copy(order="F")
    assert xk.trsm(141, uplo, 111, diag, 1.0, A, X) == 0
    xk.invalidate()
    X, B = X.astype(np.float64), B.astype(np.float64)
    norm = lambda M: np.abs(M).sum(axis=1).max()
    res = norm(T @ X - B) / ((norm(T) * norm(X) + norm(B)) * n * np.finfo(dtype).eps)
    assert res <= 10, res


@pytest.mark.parametrize("uplo", [121, 122])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_potrf_diagonal_roundings(xk, dtype, uplo):
    """The diagonal of L L^T against A at the order of a leaf, where the diagonal is
    far larger than any product: each of 7.5 pivots of its own tile, 3.5 updates by
    other tiles and the root rounds it once on average, 13 roundings of 0.42 u (u =
    eps / 2) at random, 1.5 u in the mean square; 65 roundings, with the products
    of an update added one by one, 3.4 u.  Bar 2.4 u."""
    n, e = 128, []
    for seed in range(8):
        A = spd(rng(seed), n, dtype)
        F = A.copy(order="F")
        assert xk.potrf(uplo, F) == 0
        xk.invalidate()
        L = (np.tril(F) if uplo == 122 else np.triu(F).T).astype(np.longdouble)
        d = (L * L).sum(axis=1) / np.diag(A).astype(np.longdouble) - 1
        e.append(float(np.sqrt(np.mean(d * d))))
    assert np.mean(e) <= 2.4 * np.finfo(dtype).eps / 2, e
