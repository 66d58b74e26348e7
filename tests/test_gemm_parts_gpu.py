"""Products of few tiles and a long inner dimension, which are computed in parts
of it: remainders of a part, one to 32 parts, odd and even leading dimensions,
each op, triangles, beta = 0 over NaN.  Bar: |C - ref| <= (k + 8) eps (|alpha|
|A| |B| + |beta| |C|) for each element, ref in FP64 on FP32 inputs and by a
compensated product on FP64 ones (their own rounding is inside the bar)."""
import numpy as np
import pytest

from helpers import rng

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 511), (1, 1, 512), (65, 9, 1000), (100, 100, 6149), (300, 301, 2017), (512, 500, 1199), (512, 500, 1200),
          (640, 1300, 1831)]


def _fort(r, m, n, dt):
    return np.asfortranarray(r.uniform(-1, 1, (m, n)).astype(dt))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("ops", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_gemm_in_parts(xk, m, n, k, ops, dt):
    r = rng(m + n + k)
    A = _fort(r, *((m, k) if ops[0] == "N" else (k, m)), dt)
    B = _fort(r, *((k, n) if ops[1] == "N" else (n, k)), dt)
    beta = 0.0 if ops in ("NN", "TT") else -0.75
    C = _fort(r, m, n, dt)
    C0 = C.astype(np.float64)
    if beta == 0.0:
        C[:] = np.nan
    op = {"N": xk.NoTrans, "T": xk.Trans}
    xk.gemm(op[ops[0]], op[ops[1]], 1.25, A, B, beta, C)
    xk.invalidate()
    X, Y = (M.astype(np.float64) if o == "N" else M.astype(np.float64).T for M, o in zip((A, B), ops))
    bar = (k + 8) * np.finfo(dt).eps * (1.25 * np.abs(X) @ np.abs(Y) + np.abs(beta * C0))
    assert np.all(np.abs(C - (1.25 * X @ Y + beta * C0)) <= bar)


@pytest.mark.parametrize("dt", [np.float64, np.float32, np.complex128])
@pytest.mark.parametrize("uplo", [121, 122])
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("n,k", [(1, 512), (63, 513), (300, 1000), (517, 1511), (1100, 1201)])
def test_triangle_in_parts(xk, n, k, trans, uplo, dt):
    r = rng(n + k)
    real = np.float32 if dt == np.float32 else np.float64
    A = _fort(r, *((k, n) if trans else (n, k)), real).astype(dt)
    if dt == np.complex128:
        A = np.asfortranarray(A + 1j * r.uniform(-1, 1, A.shape))
    A = np.asfortranarray(A)
    C = np.full((n, n), np.nan, dt, order="F")
    if dt == np.complex128:
        xk.herk(uplo, xk.ConjTrans if trans else xk.NoTrans, 1.25, A, 0.0, C)
    else:
        xk.syrk(uplo, xk.Trans if trans else xk.NoTrans, 1.25, A, 0.0, C)
    xk.invalidate()
    X = A.conj().T if trans else A
    X = X.astype(np.complex128 if dt == np.complex128 else np.float64)
    off = np.triu_indices(n, 1) if uplo == 122 else np.tril_indices(n, -1)
    assert np.all(np.isnan(C[off]))
    ref = 1.25 * X @ X.conj().T
    bar = (2 * k + 8) * np.finfo(real).eps * (1.25 * np.abs(X) @ np.abs(X).T)
    C[off] = ref[off]
    assert np.all(np.abs(C - ref) <= bar)


CHILD = """
import sys
sys.path.insert(0, %r)
import numpy as np, xkblas_amd as xk
L = xk.lib()
L.xkblas_init()
r = np.random.default_rng(3)
A, B = (np.asfortranarray(r.uniform(-1, 1, s)) for s in ((300, 1500), (1500, 200)))
out = []
for tile in (0, 32):  # a set tile: one part
    L.xkblas_set_gemm_tile(tile)
    C = np.zeros((300, 200), order="F")
    xk.gemm(xk.NoTrans, xk.NoTrans, 1.0, A, B, 0.0, C)
    out.append(C)
print("same" if np.array_equal(*out) else "different")
"""


@pytest.mark.parametrize("value,want", [("0", "same"), ("1", "different")])
def test_no_parts_when_switched_off(xk, value, want):
    """XKBLAS_SPLITK=0: the sums of one part, bit for bit."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    p = subprocess.run([sys.executable, "-c", CHILD % root], env=dict(os.environ, XKBLAS_SPLITK=value), timeout=60,
                       capture_output=True, text=True)
    assert p.returncode == 0 and p.stdout.strip() == want, p.stdout + p.stderr
