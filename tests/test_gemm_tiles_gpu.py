"""The product kernels at the sizes where their tiles (32, 64, 128) and stages
(16 doubles, 32 floats) end.  Small-integer operands make every product and
sum exact, so results equal NumPy's bit for bit whatever the tile; on general
operands all tiles give the same bits (the same inner order per element)."""
import numpy as np
import pytest

from helpers import rng, small_int, uniform

pytestmark = pytest.mark.gpu

OPS = [(111, 111), (111, 112), (112, 111), (112, 112)]
SHAPES = [(1, 1, 1), (31, 33, 15), (32, 64, 16), (33, 31, 17), (63, 65, 31), (64, 128, 32), (65, 127, 33),
          (127, 129, 64), (128, 128, 48), (129, 257, 65), (255, 130, 100), (260, 5, 131), (3, 300, 259), (193, 191, 1)]


@pytest.fixture(params=[0, 32, 64, 128])
def tile(request, xk):
    xk.lib().xkblas_set_gemm_tile(request.param)
    yield request.param
    xk.lib().xkblas_set_gemm_tile(0)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ta,tb", OPS)
def test_tiles_exact_on_integers(xk, tile, ta, tb, dtype):
    for M, N, K in SHAPES:
        r = rng(M * 7 + N * 3 + K)
        A = small_int(r, *((M, K) if ta == 111 else (K, M)), dtype=dtype)
        B = small_int(r, *((K, N) if tb == 111 else (N, K)), dtype=dtype)
        C = small_int(r, M, N, dtype=dtype)
        ref = 2 * (A if ta == 111 else A.T) @ (B if tb == 111 else B.T) - C
        xk.gemm(ta, tb, 2.0, A, B, -1.0, C)
        xk.invalidate()
        assert np.array_equal(C, ref), (M, N, K)


@pytest.mark.parametrize("uplo", [121, 122])
@pytest.mark.parametrize("trans", [111, 112])
def test_triangles_exact_on_integers(xk, tile, trans, uplo):
    for N, K in [(1, 5), (33, 16), (64, 40), (130, 17), (257, 100), (300, 33)]:
        r = rng(N + K)
        A = small_int(r, *((N, K) if trans == 111 else (K, N)))
        C = small_int(r, N, N)
        P = A @ A.T if trans == 111 else A.T @ A
        keep = np.triu(np.ones((N, N), bool), 1) if uplo == 122 else np.tril(np.ones((N, N), bool), -1)
        ref = np.where(keep, C, P + 3 * C)
        xk.syrk(uplo, trans, 1.0, A, 3.0, C)
        xk.invalidate()
        assert np.array_equal(C, ref), (N, K)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ta,tb", OPS)
def test_tiles_give_the_same_bits(xk, ta, tb, dtype):
    r = rng(11)
    M, N, K = 300, 201, 403
    A = uniform(r, *((M, K) if ta == 111 else (K, M)), dtype=dtype)
    B = uniform(r, *((K, N) if tb == 111 else (N, K)), dtype=dtype)
    out = []
    # a tile size of 67 rows: row panels at offsets that are not 16-byte
    # aligned, through the register-staged kernel
    for t, nb in [(32, 512), (64, 512), (128, 512), (0, 67)]:
        xk.lib().xkblas_set_gemm_tile(t)
        xk.lib().xkblas_set_param(nb, 0)
        C = np.zeros((M, N), dtype=dtype, order="F")
        xk.gemm(ta, tb, 1.0, A, B, 0.0, C)
        xk.invalidate()
        out.append(C)
    xk.lib().xkblas_set_gemm_tile(0)
    xk.lib().xkblas_set_param(0, 0)
    for C in out[1:]:
        assert np.array_equal(out[0], C)


@pytest.mark.parametrize("ta,tb", OPS)
def test_last_round_in_quarters(xk, ta, tb):
    """A little more than one round of 128 x 128 tiles: whole tiles and
    quarters together give what 64 x 64 tiles give, bit for bit."""
    r = rng(4)
    M, N, K = 2950, 2930, 2001
    A = uniform(r, *((M, K) if ta == 111 else (K, M)), dtype=np.float32)
    B = uniform(r, *((K, N) if tb == 111 else (N, K)), dtype=np.float32)
    out = []
    for t in (0, 64):
        xk.lib().xkblas_set_gemm_tile(t)
        C = np.zeros((M, N), dtype=np.float32, order="F")
        xk.gemm(ta, tb, 1.0, A, B, 0.0, C)
        xk.invalidate()
        out.append(C)
    xk.lib().xkblas_set_gemm_tile(0)
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("uplo", [121, 122])
def test_last_round_of_a_triangle_in_quarters(xk, uplo):
    A = uniform(rng(6), 4070, 2001, dtype=np.float32)
    out = []
    for t in (0, 64):
        xk.lib().xkblas_set_gemm_tile(t)
        C = np.full((4070, 4070), 7, dtype=np.float32, order="F")
        xk.syrk(uplo, 111, 1.0, A, 0.5, C)
        xk.invalidate()
        out.append(C)
    xk.lib().xkblas_set_gemm_tile(0)
    assert np.array_equal(out[0], out[1])
    assert np.all((np.triu(out[0], 1) if uplo == 122 else np.tril(out[0], -1))[np.triu_indices(4070, 1) if uplo == 122
                  else np.tril_indices(4070, -1)] == 7)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ta,tb", OPS)
def test_ring_ends_in_a_remainder_of_any_size(xk, ta, tb, dtype):
    """The ring of four stages behind 2 to 9 whole ones, with remainders that leave
    some waves nothing to load in the last: exact on integers."""
    M, N = 901, 1030
    r = rng(3)
    xk.lib().xkblas_set_gemm_tile(32)
    try:
        for K in (33, 49, 50, 52, 63, 64, 65, 97, 100, 113, 127, 129, 145, 161, 289):
            A = small_int(r, *((M, K) if ta == 111 else (K, M)), dtype=dtype)
            B = small_int(r, *((K, N) if tb == 111 else (N, K)), dtype=dtype)
            C = np.full((M, N), np.nan, dtype=dtype, order="F")
            xk.gemm(ta, tb, 1.0, A, B, 0.0, C)
            xk.invalidate()
            assert np.array_equal(C, (A if ta == 111 else A.T) @ (B if tb == 111 else B.T)), K
    finally:
        xk.lib().xkblas_set_gemm_tile(0)


@pytest.mark.parametrize("ta,tb", OPS)
@pytest.mark.parametrize("dtype,M,N,K", [
    (np.float64, 700, 901, 31), (np.float64, 700, 901, 32), (np.float64, 160, 7680, 127), (np.float64, 160, 7680, 128),
    (np.float32, 1100, 1000, 63), (np.float32, 1100, 1000, 33), (np.float32, 1100, 1000, 64),
    (np.float32, 7168, 7200, 576), (np.float32, 7100, 7300, 600)])
def test_kernel_by_rule_gives_the_same_bits(xk, dtype, M, N, K, ta, tb):
    """On both sides of the lines between the two kernels (short inner dimensions;
    FP32 over many rounds, C's columns a multiple of 4 KB apart or not): what 64 x
    64 tiles of the other kernel give, bit for bit."""
    r = rng(K)
    A = (r.random((K, M) if ta == 111 else (M, K), dtype=dtype) - dtype(0.5)).T
    B = (r.random((N, K) if tb == 111 else (K, N), dtype=dtype) - dtype(0.5)).T
    out = []
    for t in (0, 64):
        xk.lib().xkblas_set_gemm_tile(t)
        C = np.ones((N, M), dtype=dtype).T
        xk.gemm(ta, tb, 1.5, A, B, -0.5, C)
        xk.invalidate()
        out.append(C)
    xk.lib().xkblas_set_gemm_tile(0)
    assert np.array_equal(out[0], out[1])
