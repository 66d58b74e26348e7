"""Cholesky with split products, and the solve with refinement behind it, when
the program sets no block order: at the last order that the solve factors in
one block, the first that it does not, and a last block of few orders.  Bars:
||A - L L^T|| / (N ||A|| eps) <= 10 of the reference's driver, and twice the
solve's own stopping test ||b - A x|| <= ||x|| ||A|| eps sqrt(N), since the
residual is rounded once more here.  The unread triangle holds NaN."""
import numpy as np
import pytest

from helpers import rng, spd, uniform

pytestmark = pytest.mark.gpu


def _half(A, uplo):
    S = A.copy(order="F")
    S[np.triu_indices(A.shape[0], 1) if uplo == 122 else np.tril_indices(A.shape[0], -1)] = np.nan
    return S


@pytest.mark.parametrize("uplo,n", [(122, 4608), (121, 4609), (122, 4097)])
def test_posv_ir_default_order(xk, uplo, n):
    r = rng(n)
    A, B = spd(r, n), uniform(r, n, 3)
    X, info, it = xk.posv_ir(uplo, _half(A, uplo), B)
    xk.invalidate()
    assert info == 0 and it >= 1
    R = np.abs(B - A @ X).max(axis=0)
    bar = np.abs(X).max(axis=0) * np.abs(A).sum(axis=1).max() * 2.0**-53 * np.sqrt(n)
    assert np.all(R <= 2 * bar)


@pytest.mark.parametrize("mode", [2, 3])
@pytest.mark.parametrize("uplo,n", [(122, 4100), (121, 2049)])
def test_split_potrf_default_order(xk, uplo, n, mode):
    A = spd(rng(n), n)
    F = _half(A, uplo)
    xk.lib().xkblas_set_modemath(mode)
    try:
        assert xk.potrf(uplo, F) == 0
    finally:
        xk.lib().xkblas_set_modemath(0)
        xk.invalidate()
    off = np.triu_indices(n, 1) if uplo == 122 else np.tril_indices(n, -1)
    assert np.all(np.isnan(F[off]))
    F[off] = 0
    L = F if uplo == 122 else F.T
    assert np.linalg.norm(A - L @ L.T, 1) / (n * np.linalg.norm(A, 1) * 2.0**-53) <= 10


def test_leaf_beside_products_is_repeatable(xk):
    """The leaves of each block run beside the split products of the block
    before, which delays some of a leaf's waves: the factor has the same bits
    every time."""
    n, L = 4096, xk.lib()
    A = spd(rng(7), n)
    first = None
    nb0 = L.xkblas_get_param()
    L.xkblas_set_modemath(2)
    L.xkblas_set_param(1024, 0)
    try:
        for _ in range(12):
            F = A.copy(order="F")
            assert xk.potrf(122, F) == 0
            xk.invalidate()
            first = F if first is None else first
            assert np.array_equal(F, first)
    finally:
        L.xkblas_set_modemath(0)
        L.xkblas_set_param(nb0, 0)
        xk.invalidate()
