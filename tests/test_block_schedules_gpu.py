"""The blocked factorizations and solves that the default mode's smaller orders
do not take: Cholesky in blocks of NB with split products (paired trailing updates
and one per panel; complex), and the complex factorization and left solve beyond
the order up to which they run as real ones of twice the order.  Even and odd
block counts, ragged last blocks, a failing pivot behind every deferred update;
bars of the reference's drivers."""
import numpy as np
import pytest

from helpers import rng, spd

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[2, 3])
def split(xk, request):
    xk.lib().xkblas_set_modemath(request.param)
    yield request.param
    xk.lib().xkblas_set_modemath(0)
    xk.lib().xkblas_set_param(0, 0)
    xk.lib().xkblas_set_potrf_pairing(-1)


@pytest.mark.parametrize("uplo", [121, 122])
@pytest.mark.parametrize("pairing", [0, 1])
@pytest.mark.parametrize("n,nb", [(1000, 128), (1100, 256), (640, 128), (513, 64), (300, 256)])
def test_split_potrf_schedules(xk, orc, split, uplo, pairing, n, nb):
    L = xk.lib()
    A0 = spd(rng(n + nb), n)
    L.xkblas_set_param(nb, 0)
    L.xkblas_set_potrf_pairing(pairing)
    A = A0.copy(order="F")
    assert xk.potrf(uplo, A) == 0
    xk.invalidate()
    assert orc.potrf_residual(A0, A, uplo) <= 10.0
    other = np.triu_indices(n, 1) if uplo == 122 else np.tril_indices(n, -1)
    assert np.array_equal(A[other], A0[other])
    bad = n - 1 - (n % nb or nb) // 2  # inside the last block
    A = A0.copy(order="F")
    A[bad, bad] = -1e6
    assert xk.potrf(uplo, A) == bad + 1
    xk.invalidate()


@pytest.mark.parametrize("uplo", [121, 122])
@pytest.mark.parametrize("n,nb", [(300, 128), (777, 256), (512, 128), (129, 64)])
def test_split_zpotrf_blocks(xk, split, uplo, n, nb):
    r = rng(n + uplo)
    G = r.uniform(-0.5, 0.5, (n, n)) + 1j * r.uniform(-0.5, 0.5, (n, n))
    H = np.asfortranarray(G @ G.conj().T + n * np.eye(n))
    xk.lib().xkblas_set_param(nb, 0)
    A = H.copy(order="F")
    assert xk.potrf(uplo, A) == 0
    xk.invalidate()
    F = np.tril(A) if uplo == 122 else np.triu(A).conj().T
    norm = lambda M: np.abs(M).sum(axis=1).max()
    assert norm(H - F @ F.conj().T) / (n * norm(H) * 2.0 ** -53) <= 10.0
    assert np.all(F.diagonal().imag == 0)
    other = np.triu_indices(n, 1) if uplo == 122 else np.tril_indices(n, -1)
    assert np.array_equal(A[other], H[other])
    for bad in (0, n - 1 - (n % nb or nb) // 2, n - 1):
        A = H.copy(order="F")
        A[bad, bad] = -1e6
        assert xk.potrf(uplo, A) == bad + 1
        xk.invalidate()


@pytest.mark.parametrize("uplo", [121, 122])
def test_complex_blocks_beyond_the_real_form(xk, uplo):
    """Order 8300 in nine blocks of 1024: the factor, both solves with it (left)
    and a failing pivot in the last block, by products with a few vectors."""
    n, r = 8300, rng(uplo)
    z = lambda m, k: (r.random((k, m, 2), dtype=np.float32) - np.float32(0.5)).view(np.complex64)[..., 0].T
    H = z(n, n)
    H += H.conj().T
    H[np.diag_indices(n)] = 4 * np.sqrt(n)
    V = np.asfortranarray(z(n, 5))
    HV = H @ V
    xk.lib().xkblas_set_param(1024, 0)
    try:
        A = H.copy(order="F")
        assert xk.potrf(uplo, A) == 0
        low = uplo == 122
        F = np.tril(A) if low else np.triu(A)
        eps, norm = np.finfo(np.float32).eps, np.abs(H).sum(axis=0).max()
        W = F @ (F.conj().T @ V) if low else F.conj().T @ (F @ V)
        assert np.abs(HV - W).max() <= 10 * n * eps * norm * np.abs(V).max()
        normF = np.abs(F).sum(axis=1).max()
        for op in (111, 113, 112):
            X = V.copy(order="F")
            xk.trsm(141, uplo, op, 131, np.complex64(0.5 - 1j), A, X)
            FX = (F if op == 111 else F.T if op == 112 else F.conj().T) @ X
            assert np.abs(FX - (0.5 - 1j) * V).max() <= 10 * n * eps * (normF * np.abs(X).max() + np.abs(V).max())
        xk.invalidate()
        A = H.copy(order="F")
        A[n - 50, n - 50] = -1
        assert xk.potrf(uplo, A) == n - 49
    finally:
        xk.lib().xkblas_set_param(0, 0)
        xk.invalidate()
