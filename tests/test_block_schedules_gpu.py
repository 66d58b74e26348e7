"""Cholesky in blocks of NB with split products, which the default mode does not
take: paired trailing updates and one per panel, even and odd block counts, ragged
last blocks, a failing pivot behind every deferred update; bars of the reference's
drivers."""
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
