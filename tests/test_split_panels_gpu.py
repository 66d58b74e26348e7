"""Split products of resident operands in column panels of unequal last width,
where the panels take more rounds of tiles than one launch: the same bits, copied
back while later panels run."""
import numpy as np
import pytest

from helpers import rng, uniform

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [2, 3])
@pytest.mark.parametrize("M,N,K", [(2430, 2059, 1300), (1100, 4097, 900), (4843, 1537, 1100)])
def test_split_product_in_panels(xk, M, N, K, mode):
    r = rng(M + mode)
    A, B = uniform(r, M, K), uniform(r, K, N)
    L = xk.lib()
    L.xkblas_set_modemath(mode)
    out = []
    try:
        for pipeline in (0, 1):
            L.xkblas_set_pipeline(pipeline)
            C = np.zeros((M, N), order="F")
            xk.gemm(xk.NoTrans, xk.NoTrans, 1.5, A, B, 0.0, C)
            xk.gemm(xk.NoTrans, xk.NoTrans, 0.5, A, B, -0.25, C)  # resident
            out.append(C)
            xk.invalidate()
    finally:
        L.xkblas_set_pipeline(1)
        L.xkblas_set_modemath(0)
    assert np.array_equal(out[0], out[1])
