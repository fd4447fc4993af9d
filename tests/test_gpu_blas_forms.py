"""uvt_dgemm and uvt_dtrmm on the MI355X in every tile shape: each transpose,
side, triangle and diagonal at sizes that pick wave tiles and 32x128, 128x32,
64x64, 128x128 and 256x128 workgroup tiles with ragged edges, odd leading dimensions, and NaN in
everything that is not an operand.  Small-integer inputs and power-of-two
factors make every sum exact, so results equal NumPy's bit for bit."""
import ctypes as c
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L(uvt, gpu):
    lib = uvt.lib()
    lib.uvt_dtrmm.argtypes = [c.c_void_p, c.c_int, c.c_int, c.c_int, c.c_int, c.c_int64, c.c_int64, c.c_double,
                              c.c_void_p, c.c_int64, c.c_void_p, c.c_int64, c.c_void_p]
    lib.uvt_dgemm.argtypes = [c.c_void_p, c.c_int, c.c_int, c.c_int64, c.c_int64, c.c_int64, c.c_double, c.c_void_p,
                              c.c_int64, c.c_void_p, c.c_int64, c.c_double, c.c_void_p, c.c_int64, c.c_void_p]
    lib.uvt_dtrmm.restype = lib.uvt_dgemm.restype = c.c_int
    return lib


def padded(x, pad, fill=np.nan):
    y = np.full((x.shape[0], x.shape[1] + pad), fill)
    y[:, :x.shape[1]] = x
    return y


FORMS = list(itertools.product((0, 1), (0, 1), (0, 1), (0, 1)))  # side, uplo, trans, diag
BIG = [(0, 0, 0, 0), (0, 1, 0, 1), (0, 0, 1, 1), (0, 1, 1, 0), (1, 0, 0, 1), (1, 1, 1, 1), (1, 0, 1, 0), (1, 1, 0, 0)]
CASES = [(f, s) for f in FORMS for s in ((1, 1), (40, 301), (301, 40), (257, 131), (700, 633))] + \
        [(f, (1901, 1802)) for f in BIG] + [(f, (2900, 2951)) for f in BIG] + \
        [((0, 0, 1, 0), (12300, 41)), ((1, 1, 0, 1), (41, 12300))] + \
        [(f, s) for f in BIG for s in ((1200, 1207), (1601, 1500))] + [(f, (4096, 4096)) for f in ((0, 1, 0, 0), (1, 1, 1, 1))]


@pytest.mark.parametrize("form,size", CASES)
def test_dtrmm_exact(L, gpu, form, size):
    (side, uplo, trans, diag), (m, n) = form, size
    rng = np.random.default_rng(m * 7 + n)
    nt = n if side else m
    T = rng.integers(-2, 3, (nt, nt)).astype(np.float64)
    keep = np.triu(np.ones((nt, nt), bool)) if uplo else np.tril(np.ones((nt, nt), bool))
    if diag:
        np.fill_diagonal(keep, False)
    A = padded(np.where(keep, T, np.nan), 1)
    T = np.where(keep, T, 0.0)
    if diag:
        np.fill_diagonal(T, 1.0)
    B = rng.integers(-2, 3, (m, n)).astype(np.float64)
    op = T.T if trans else T
    want = -2.0 * (B @ op if side else op @ B)
    print("[gpu-blas] dtrmm", form, size, flush=True)
    dA, dB = gpu.array(A), gpu.array(padded(B, 3, 7.5))
    st = L.uvt_dtrmm(gpu.ptr, side, uplo, trans, diag, m, n, -2.0, dA.ptr, nt + 1, dB.ptr, n + 3, gpu.stream)
    gpu.sync()
    got = dB.download((m, n + 3))
    dA.free()
    dB.free()
    assert st == 0
    np.testing.assert_array_equal(got[:, :n], want)
    assert (got[:, n:] == 7.5).all()


@pytest.mark.parametrize("ta,tb", list(itertools.product((0, 1), (0, 1))))
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (40, 301, 65), (301, 40, 33), (257, 131, 70), (700, 633, 1),
                                   (513, 1031, 259), (1500, 1601, 200), (40001, 43, 35), (2950, 2951, 129)])
def test_dgemm_exact(L, gpu, m, n, k, ta, tb):
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    A = rng.integers(-3, 4, (k, m) if ta else (m, k)).astype(np.float64)
    B = rng.integers(-3, 4, (n, k) if tb else (k, n)).astype(np.float64)
    C = rng.integers(-3, 4, (m, n)).astype(np.float64)
    prod = (A.T if ta else A) @ (B.T if tb else B)
    for alpha, beta in ((1.0, 0.0), (-2.0, 0.5)):
        print("[gpu-blas] dgemm", (m, n, k), (ta, tb), alpha, beta, flush=True)
        dA, dB = gpu.array(padded(A, 1)), gpu.array(padded(B, 2))
        dC = gpu.array(padded(C if beta else np.full((m, n), np.nan), 3, 7.5))
        st = L.uvt_dgemm(gpu.ptr, ta, tb, m, n, k, alpha, dA.ptr, A.shape[1] + 1, dB.ptr, B.shape[1] + 2, beta,
                         dC.ptr, n + 3, gpu.stream)
        gpu.sync()
        got = dC.download((m, n + 3))
        for x in (dA, dB, dC):
            x.free()
        assert st == 0
        np.testing.assert_array_equal(got[:, :n], alpha * prod + (beta * C if beta else 0.0))
        assert (got[:, n:] == 7.5).all()
