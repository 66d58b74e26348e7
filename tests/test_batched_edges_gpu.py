"""Batched products and solves at the edges of their tiles (16, 32, 64), slices
(32) and strips (16), odd leading dimensions, with NaN in everything that is not
an operand.  Bars: GEMM |C - ref| <= (k + 4) eps (|alpha| |A| |B| + |beta| |C|)
for each element; TRSM max |alpha B - L X| <= (m + 4) eps (|L| |X| + |alpha B|)
for each element, the backward error of a substitution."""
import ctypes

import numpy as np
import pytest

from helpers import rng

pytestmark = pytest.mark.gpu


def _run(xk, problems):
    arr = (xk.BatchProblem * len(problems))(*problems)
    plan = xk.lib().xkblas_batch_create(ctypes.cast(arr, ctypes.c_void_p), len(arr))
    assert xk.lib().xkblas_batch_run(plan) == 0
    xk.lib().xkblas_sync()
    xk.lib().xkblas_batch_destroy(plan)


def _padded(M, dt, pad=3):
    """A device matrix with `pad` more rows of NaN under each column but the last."""
    m, n = M.shape
    buf = np.full((m + pad, n), np.nan, dt, order="F")
    buf[:m] = M
    flat = buf.ravel(order="F")[: (m + pad) * (n - 1) + m] if n else buf.ravel()
    return np.asfortranarray(flat.reshape(-1, 1))


def _back(D, m, n, pad=3):
    flat = D.download().ravel(order="F")
    buf = np.full((m + pad) * n, np.nan, flat.dtype)
    buf[: flat.size] = flat
    return buf.reshape((m + pad, n), order="F")


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n", [1, 16, 17, 33, 64, 65, 100])
def test_batched_trsm_edges(xk, n, dt):
    r = rng(n)
    eps = np.finfo(dt).eps
    work = []
    for m in (1, 2, 15, 16, 17, 31, 33, 48, 49, 63, 64, 65, 80, 127, 128, 129, 191, 193, 257):
        L = np.tril(r.uniform(-0.5, 0.5, (m, m))).astype(dt)
        L[np.arange(m), np.arange(m)] = np.sign(r.uniform(-1, 1, m)) * (1 + m / 8)
        B = r.uniform(-1, 1, (m, n)).astype(dt)
        S = L.copy()
        S[np.triu_indices(m, 1)] = np.nan
        dL, dB = xk.DeviceArray(_padded(S, dt)), xk.DeviceArray(_padded(B, dt))
        work.append((m, L, B, dL, dB))
    code = 0 if dt == np.float64 else 1
    _run(xk, [xk.BatchProblem(xk.BATCH_TRSM, code, xk.NoTrans, xk.NoTrans, m, n, m, 1.25, 0.0, dL.ptr, m + 3, None, 0,
                              dB.ptr, m + 3) for m, L, B, dL, dB in work])
    for m, L, B, dL, dB in work:
        X = _back(dB, m, n)
        assert np.all(np.isnan(X[m:])), m
        X, L, B = X[:m].astype(np.float64), L.astype(np.float64), 1.25 * B.astype(np.float64)
        bar = (m + 4) * eps * (np.abs(L) @ np.abs(X) + np.abs(B))
        assert np.all(np.abs(B - L @ X) <= bar), m


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("ops", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("beta", [0.0, -0.5])
def test_batched_gemm_edges(xk, ops, beta, dt):
    r = rng(5)
    eps = np.finfo(dt).eps
    work = []
    for k in (0, 1, 3, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 97):
        for m, n in ((1, 1), (31, 65), (33, 64), (64, 32), (65, 17), (129, 66)):
            A, B = r.uniform(-1, 1, (m, k)).astype(dt), r.uniform(-1, 1, (k, n)).astype(dt)
            C = r.uniform(-1, 1, (m, n)).astype(dt) if beta else np.full((m, n), np.nan, dt)
            sA, sB = (A if ops[0] == "N" else A.T), (B if ops[1] == "N" else B.T)
            dA, dB = (xk.DeviceArray(_padded(S, dt) if k else np.zeros((1, 1), dt, order="F")) for S in (sA, sB))
            work.append((A, B, C, dA, dB, xk.DeviceArray(_padded(C, dt)), sA.shape[0] + 3, sB.shape[0] + 3))
    code = 0 if dt == np.float64 else 1
    op = {"N": xk.NoTrans, "T": xk.Trans}
    _run(xk, [xk.BatchProblem(xk.BATCH_GEMM, code, op[ops[0]], op[ops[1]], A.shape[0], B.shape[1], A.shape[1], 1.5, beta,
                              dA.ptr, la, dB.ptr, lb, dC.ptr, C.shape[0] + 3) for A, B, C, dA, dB, dC, la, lb in work])
    for A, B, C, dA, dB, dC, la, lb in work:
        (m, k), n = A.shape, B.shape[1]
        got = _back(dC, m, n)
        assert np.all(np.isnan(got[m:]))
        A, B, C = (x.astype(np.float64) for x in (A, B, C if beta else np.zeros_like(C)))
        bar = (k + 4) * eps * (1.5 * np.abs(A) @ np.abs(B) + np.abs(beta * C))
        assert np.all(np.abs(got[:m] - (1.5 * A @ B + beta * C)) <= bar), (m, n, k)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_batched_trsm_keeps_rows_above_a_singular_one(xk, dt):
    m, n, bad = 70, 20, 21
    r = rng(3)
    L = np.tril(r.uniform(0.1, 0.5, (m, m))).astype(dt) + (2 * np.eye(m)).astype(dt)
    L[bad, bad] = 0
    B = r.uniform(0.5, 1, (m, n)).astype(dt)
    dL, dB = xk.DeviceArray(np.asfortranarray(L)), xk.DeviceArray(np.asfortranarray(B))
    code = 0 if dt == np.float64 else 1
    _run(xk, [xk.BatchProblem(xk.BATCH_TRSM, code, xk.NoTrans, xk.NoTrans, m, n, m, 1.0, 0.0, dL.ptr, m, None, 0, dB.ptr, m)])
    X = dB.download()
    assert np.all(np.isfinite(X[:bad])) and not np.any(np.isfinite(X[bad:]))
