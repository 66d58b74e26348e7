"""Products of resident operands in column panels and in one launch: the same
bits, at sizes where the panels are taken (several rounds over the chip, a last
panel of another tile) and where they must not be (parts of the inner dimension,
whose partial results have one place)."""
import numpy as np
import pytest

from helpers import rng

pytestmark = pytest.mark.gpu


def _mat(r, m, n, dtype):
    return np.asfortranarray(r.random((n, m), dtype=dtype).T - dtype(0.5))


@pytest.mark.parametrize("dtype,mode,op,m,n,k,beta", [
    (np.float64, 0, "NN", 4100, 4200, 2600, -0.5), (np.float64, 0, "TT", 5003, 3001, 4003, 0.0),
    (np.float32, 0, "NT", 6000, 6100, 3000, -0.5), (np.float32, 0, "TN", 4096, 4100, 1500, 0.0),
    (np.float64, 3, "NT", 8192, 5400, 3000, -0.5),
    (np.float64, 0, "NN", 15411, 158, 8000, 0.0), (np.float64, 0, "TT", 15411, 158, 3000, -0.5)])
def test_panels_equal_one_launch(xk, dtype, mode, op, m, n, k, beta):
    r = rng(m + k)
    A = _mat(r, *((m, k) if op[0] == "N" else (k, m)), dtype)
    B = _mat(r, *((k, n) if op[1] == "N" else (n, k)), dtype)
    C0 = _mat(r, m, n, dtype)
    ops = {"N": xk.NoTrans, "T": xk.Trans}
    L = xk.lib()
    xk.invalidate()
    L.xkblas_set_modemath(mode)
    L.xkblas_set_split_count(20 if mode else 0)  # 38 planes: 104 rounds
    out = []
    try:
        for pipeline in (0, 1):
            L.xkblas_set_pipeline(pipeline)
            C = C0.copy(order="F")
            D = np.zeros((m, n), dtype, order="F")
            xk.gemm(ops[op[0]], ops[op[1]], 1.0, A, B, 0.0, D)  # operands from the host
            xk.gemm(ops[op[0]], ops[op[1]], 1.5, A, B, beta, C, sync=False)
            xk.gemm(ops[op[0]], ops[op[1]], 1.5, A, B, beta, C)  # all resident
            out.append((D.copy(), C))
            xk.gemm(ops[op[0]], ops[op[1]], 1.0, A, B, 0.0, D)  # all resident
            assert np.array_equal(D, out[-1][0])
            xk.invalidate()
    finally:
        L.xkblas_set_pipeline(1)
        L.xkblas_set_modemath(0)
        L.xkblas_set_split_count(0)
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
