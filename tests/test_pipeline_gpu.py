"""Row-panel pipelining of products whose operands start in host memory.

A DGEMM whose op(A) or C is not yet on the device runs one tile row of C at
a time, each panel waiting only for its own copies, and the copy back of C
follows the panels.  Every element sees the same operands and inner order
as the single launch of the resident path, so the results must be equal bit
for bit, in FP64 MFMA and in the split modes (row scalings span the whole
inner dimension; B's residue planes are computed once), for ragged shapes,
every transpose pair and beta = 0 (C not read) or not.
"""
import ctypes

import numpy as np
import pytest

from helpers import rng, uniform

pytestmark = pytest.mark.gpu

N_, T_ = 111, 112


def _run(xk, pipeline, ta, tb, alpha, A, B, beta, C0, nb):
    L = xk.lib()
    xk.invalidate()
    L.xkblas_set_param(nb, 0)
    L.xkblas_set_pipeline(pipeline)
    try:
        C = C0.copy(order="F")
        assert xk.gemm(ta, tb, alpha, A, B, beta, C) == 0
    finally:
        L.xkblas_set_pipeline(1)
        xk.invalidate()
    return C


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("ta,tb", [(N_, N_), (T_, N_), (N_, T_), (T_, T_)])
@pytest.mark.parametrize("beta", [0.0, -0.5])
def test_pipelined_equals_one_launch(xk, orc, mode, ta, tb, beta):
    M, N, K, nb = 700, 300, 500, 128
    r = rng(31 + ta + 2 * tb + (beta != 0) + 7 * mode)
    A = uniform(r, M, K) if ta == N_ else uniform(r, K, M)
    B = uniform(r, K, N) if tb == N_ else uniform(r, N, K)
    C0 = uniform(r, M, N)
    L = xk.lib()
    L.xkblas_set_modemath(mode)
    try:
        Cp = _run(xk, 1, ta, tb, 1.5, A, B, beta, C0, nb)
        Cr = _run(xk, 0, ta, tb, 1.5, A, B, beta, C0, nb)
    finally:
        L.xkblas_set_modemath(0)
    assert np.array_equal(Cp, Cr)
    Cref = orc.dgemm_tiled(ta, tb, 1.5, A, B, beta, C0.copy(order="F"), nb)
    assert orc.gemm_residual(1.5, A, B, beta, C0, Cref, Cp) <= 3.0


def test_pipelined_then_resident_reuse(xk):
    """A pipelined product leaves its operands resident: the same call again
    (one launch, nothing to fetch) gives the same bits, and a partial copy
    back of C (rows of two panels) waits only for the panels it reads."""
    M, N, K, nb = 1000, 260, 300, 256
    r = rng(41)
    A, B, C0 = uniform(r, M, K), uniform(r, K, N), uniform(r, M, N)
    L = xk.lib()
    xk.invalidate()
    L.xkblas_set_param(nb, 0)
    C = C0.copy(order="F")
    Cs = C0.copy(order="F")
    xk.gemm(N_, N_, 1.0, A, B, 0.0, C, sync=False)
    L.xkblas_memory_coherent_async(0, 0, 300, N, C.ctypes.data, M, 8)
    L.xkblas_sync()
    top = C[:300].copy()
    xk.coherent(C)
    xk.gemm(N_, N_, 1.0, A, B, 0.0, Cs)
    xk.invalidate()
    assert np.array_equal(top, C[:300])
    assert np.array_equal(C, Cs)
    np.testing.assert_allclose(C, A @ B, rtol=0, atol=1e-12)


@pytest.mark.parametrize("ta,tb", [(N_, N_), (T_, N_), (N_, T_), (T_, T_)])
@pytest.mark.parametrize("mode,dtype", [(0, np.float64), (0, np.float32), (2, np.float64)])
def test_resident_product_in_panels_equals_one_launch(xk, ta, tb, mode, dtype):
    """A large result of resident operands is computed in column panels so
    that its copy back runs beside the product: the same bits as one launch,
    for a whole copy back, a part of it first, and a second product that
    follows before the copy back (which then reads and waits correctly)."""
    M, N, K = 2000, 2900 if dtype == np.float32 else 1900, 600
    r = rng(5 + ta + 2 * tb + mode)
    A = uniform(r, *((M, K) if ta == N_ else (K, M)), dtype=dtype)
    B = uniform(r, *((K, N) if tb == N_ else (N, K)), dtype=dtype)
    L = xk.lib()
    xk.invalidate()
    L.xkblas_set_param(700, 0)
    L.xkblas_set_modemath(mode)
    out = []
    try:
        for pipeline in (0, 1):
            L.xkblas_set_pipeline(pipeline)
            C, D = np.zeros((M, N), dtype, order="F"), np.zeros((M, 40), dtype, order="F")
            E = uniform(rng(9), N, 40, dtype=dtype)
            for beta in (0.0, -0.5):
                xk.gemm(ta, tb, 1.5, A, B, beta, C, sync=False)
            xk.gemm(N_, N_, 1.0, C, E, 0.0, D, sync=False)
            L.xkblas_memory_coherent_async(0, 0, 300, 1000, C.ctypes.data, M, C.itemsize)
            L.xkblas_sync()
            top = C[:300, :1000].copy()
            xk.coherent(C)
            xk.coherent(D)
            xk.gemm(ta, tb, 1.0, A, B, 0.0, C)  # all operands resident, copied back at once
            out.append((top, D, C))
            xk.invalidate()
    finally:
        L.xkblas_set_pipeline(1)
        L.xkblas_set_modemath(0)
        L.xkblas_set_param(0, 0)
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_copies_back_of_short_and_long_calls(xk):
    """Results of short calls (copied back behind the whole stream) and long ones
    (behind their own event), with calls of the other kind between and a mirror
    written by both in turn: exact on integers."""
    n = 2400
    r = rng(8)
    A = np.asfortranarray(r.integers(-2, 3, (n, n)).astype(np.float64))
    a = np.asfortranarray(r.integers(-2, 3, (n, 20)).astype(np.float64))
    long_, short = A @ A, a @ a.T
    C, D, E = (np.zeros((n, n), order="F") for _ in range(3))
    for _ in range(3):
        xk.gemm(N_, T_, 1.0, a, a, 0.0, C, sync=False)   # short
        xk.gemm(N_, N_, 1.0, A, A, 0.0, D, sync=False)   # long
        xk.gemm(N_, T_, 1.0, a, a, 0.0, E, sync=False)
        xk.coherent(C)
        assert np.array_equal(C, short)
        xk.gemm(N_, N_, 1.0, A, A, 1.0, E, sync=False)   # the same mirror, long
        xk.coherent(D)
        assert np.array_equal(D, long_)
        xk.gemm(N_, T_, 1.0, a, a, 1.0, E, sync=False)   # and short
        xk.gemm(N_, N_, 1.0, A, A, 0.0, C, sync=False)
        xk.coherent(E)
        xk.coherent(C)
        assert np.array_equal(E, long_ + 2 * short)
        assert np.array_equal(C, long_)
    xk.invalidate()


@pytest.mark.parametrize("follows", ["gemm", "syr2k"])
def test_copy_back_of_a_short_calls_result_runs_under_the_next_call(xk, follows, tmp_path):
    """A result waits for its own last write: its copy back (0.3 ms) ends while a
    long call (2 ms and more) that was enqueued after it still runs, also where a
    short call stands between."""
    import csv
    L = xk.lib()
    n, m = 1500, 4200
    r = rng(9)
    a = np.asfortranarray(r.integers(-2, 3, (n, 20)).astype(np.float64))
    A = np.asfortranarray(r.integers(-2, 3, (m, m)).astype(np.float64))
    s = np.asfortranarray(r.integers(-2, 3, (40, 20)).astype(np.float64))
    p = L.xkblas_malloc(n * n * 8)
    buf = (ctypes.c_double * (n * n)).from_address(p)
    C = np.frombuffer(buf).reshape((n, n), order="F")
    D, E = np.zeros((m, m), order="F"), np.zeros((40, 40), order="F")

    def calls():
        xk.gemm(N_, T_, 1.0, a, a, 0.0, C, sync=False)
        xk.gemm(N_, T_, 1.0, s, s, 0.0, E, sync=False)
        if follows == "gemm":
            xk.gemm(N_, N_, 1.0, A, A, 0.0, D, sync=False)
        else:
            xk.syr2k(122, N_, 1.0, A, A, 0.0, D, sync=False)

    try:
        calls()
        L.xkblas_sync()  # the operands are resident
        C[:] = 0
        assert L.xkblas_trace_start(str(tmp_path).encode()) == 0
        calls()
        L.xkblas_memory_coherent_async(0, 0, n, n, C.ctypes.data, n, 8)
        L.xkblas_sync()
        assert L.xkblas_trace_stop() == 0
        assert np.array_equal(C, a @ a.T)
        with open(tmp_path / "kern.csv") as f:
            kern = list(csv.DictReader(f))
        with open(tmp_path / "cpy.csv") as f:
            back = [c for c in csv.DictReader(f) if c["Dir"] == "2"]
        assert sum(int(c["Size"]) for c in back) == n * n * 8
        assert max(float(c["End"]) for c in back) < float(kern[-1]["End"])
    finally:
        xk.invalidate()
        L.xkblas_free(p, n * n * 8)
