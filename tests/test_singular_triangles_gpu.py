"""Solves with a zero or NaN on the diagonal: as in a substitution, the
solutions before that row (behind it, for the other direction) are finite and
those of the triangle without it.  Positions at the ends of a 16 x 16 tile, of a
leaf of 128 and of a block.  Bar: 10 n eps on entries of size one (diagonal 1.5,
entries below 1 / n)."""
import numpy as np
import pytest
from scipy.linalg import solve_triangular

from helpers import rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128, np.complex64])
@pytest.mark.parametrize("uplo", [121, 122])
@pytest.mark.parametrize("trans", [111, 112])
@pytest.mark.parametrize("bad,value", [(9, 0.0), (9, np.nan), (15, 0.0), (16, 0.0), (73, 0.0), (127, np.nan), (130, 0.0), (259, 0.0)])
def test_rows_before_a_singular_pivot(xk, bad, value, trans, uplo, dtype):
    n = 300
    r = rng(bad + uplo + trans)
    A = r.uniform(-0.5, 0.5, (n, n)) / n
    if np.dtype(dtype).kind == "c":
        A = A + 1j * r.uniform(-0.5, 0.5, (n, n)) / n
    A = np.asfortranarray(A.astype(dtype))
    A[np.diag_indices(n)] = 1.5
    A[bad, bad] = value
    B = np.asfortranarray(r.uniform(-1, 1, (n, 5)).astype(dtype))
    X = B.copy(order="F")
    xk.trsm(141, uplo, trans, 131, 1.0, A, X)
    xk.invalidate()
    forward = (uplo == 122) == (trans == 111)
    rows = slice(0, bad) if forward else slice(bad + 1, n)
    ref = solve_triangular(A[rows, rows].astype(np.complex128), B[rows], lower=uplo == 122, trans=0 if trans == 111 else 1)
    assert np.all(np.abs(X[rows] - ref) <= 10 * n * np.finfo(dtype).eps)
