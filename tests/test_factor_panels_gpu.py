"""Cholesky at the order up to which it is one block column on one stream, and
beyond it, in block columns of 512 on two streams (whole ones, and a last one of
one order), with the reference driver's bar ||A - L L^T|| / (N ||A|| eps) <= 10.
The unread triangle holds NaN and keeps it; a failing pivot is found beyond the
first block columns."""
import numpy as np
import pytest

from helpers import rng, spd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("uplo,n", [(122, 4608), (121, 4609), (122, 5120), (121, 5121)])
def test_potrf_one_block_column_or_many(xk, n, uplo, dtype):
    A = spd(rng(n), n, dtype)
    off = np.triu_indices(n, 1) if uplo == 122 else np.tril_indices(n, -1)
    F = A.copy(order="F")
    F[off] = np.nan
    assert xk.potrf(uplo, F) == 0
    xk.invalidate()
    assert np.all(np.isnan(F[off]))
    F[off] = 0
    L = (F if uplo == 122 else F.T).astype(np.float64)
    A = A.astype(np.float64)
    eps = np.finfo(dtype).eps / 2
    assert np.linalg.norm(A - L @ L.T, 1) / (n * np.linalg.norm(A, 1) * eps) <= 10


@pytest.mark.parametrize("uplo,n,bad", [(122, 4608, 4000), (121, 4700, 4690)])
def test_potrf_finds_a_late_pivot(xk, n, uplo, bad):
    A = np.asfortranarray(np.eye(n) * 4 + 1e-3)
    A[bad, bad] = -1
    assert xk.potrf(uplo, A) == bad + 1
    xk.invalidate()
