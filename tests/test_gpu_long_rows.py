"""Operands whose rows lie 16 MB to 268 MB apart on the MI355X, past the 32-bit
offsets of the steady state: wave tiles, whole 64x64, 128x128 and 256x128
tiles, cut and stream-K reductions, a dgemm and a dtrmm.  Small-integer inputs
make every sum exact in any order, so results equal NumPy's bit for bit."""
import ctypes as c

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def strided(gpu, x, ld, pad=8):
    """x in rows of ld elements on the device, NaN behind each row's end."""
    rows, cols = x.shape
    host = np.full((rows, cols + pad), np.nan)
    host[:, :cols] = x
    b = gpu.alloc(((rows - 1) * ld + cols + pad) * 8)
    b.upload_2d(host, (cols + pad) * 8, rows, ld * 8, (cols + pad) * 8)
    return b


@pytest.mark.parametrize("n,m,lda,ldb,form", [
    (61, 50, (1 << 24) + 1, (1 << 24) + 3, "whole"),    # wave tiles, both operands
    (300, 3001, (1 << 24) + 1, 3009, "whole"),          # 16x32 wave tiles
    (513, 6401, (1 << 23) + 1, 6409, "whole"),          # 64x64
    (1290, 2700, (1 << 23) + 1, 2708, "cut"),           # 64x64, cut
    (520, 16000, (1 << 22) + 1, 16009, "whole"),        # 128x128
    (600, 14000, (1 << 22) + 1, 14008, "cut"),          # stream-K
    (1024, 16384, (1 << 21) + 1, 16392, "whole"),       # 256x128
])
def test_trmm_of_long_rows(gpu, uvt, n, m, lda, ldb, form):
    rng = np.random.default_rng(n + m)
    A = rng.integers(-2, 3, (n, n)).astype(np.float64)
    B = rng.integers(-2, 3, (n, m)).astype(np.float64)
    want = np.tril(A) @ B
    A[np.triu_indices(n, 1)] = np.nan
    plan = uvt.Plan(n, m)
    wg, parts = gpu.plan_launch_info(plan)
    print("[gpu-long-rows] trmm", n, m, lda, ldb, wg, parts, flush=True)
    assert (parts > 0) == (form == "cut")
    dA, dB, dC = strided(gpu, A, lda), strided(gpu, B, ldb), gpu.alloc(n * m * 8)
    try:
        gpu.trmm_f64(plan, dA, lda, dB, ldb, dC, m)
        gpu.sync()
        np.testing.assert_array_equal(dC.download((n, m)), want)
    finally:
        plan.close()
        for b in (dA, dB, dC):
            b.free()


@pytest.mark.parametrize("m,n,k", [(70, 130, 90), (40, 1030, 33)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_dgemm_of_long_rows(gpu, uvt, m, n, k, ta, tb):
    L = uvt.lib()
    L.uvt_dgemm.argtypes = [c.c_void_p, c.c_int, c.c_int, c.c_int64, c.c_int64, c.c_int64, c.c_double, c.c_void_p,
                            c.c_int64, c.c_void_p, c.c_int64, c.c_double, c.c_void_p, c.c_int64, c.c_void_p]
    rng = np.random.default_rng(m + n + k)
    A = rng.integers(-3, 4, (k, m) if ta else (m, k)).astype(np.float64)
    B = rng.integers(-3, 4, (n, k) if tb else (k, n)).astype(np.float64)
    ld = (1 << 25) + 1 if not tb else (1 << 22) + 1
    print("[gpu-long-rows] dgemm", (m, n, k), ta, tb, flush=True)
    dA, dB, dC = strided(gpu, A, (1 << 24) + 1), strided(gpu, B, ld), gpu.alloc(m * n * 8)
    try:
        st = L.uvt_dgemm(gpu.ptr, ta, tb, m, n, k, 1.0, dA.ptr, (1 << 24) + 1, dB.ptr, ld, 0.0, dC.ptr, n, gpu.stream)
        gpu.sync()
        assert st == 0
        np.testing.assert_array_equal(dC.download((m, n)), (A.T if ta else A) @ (B.T if tb else B))
    finally:
        for b in (dA, dB, dC):
            b.free()


@pytest.mark.parametrize("side,uplo,trans,diag", [(0, 0, 0, 0), (0, 1, 1, 1), (1, 0, 1, 0), (1, 1, 0, 1)])
def test_dtrmm_of_long_rows(gpu, uvt, side, uplo, trans, diag):
    L = uvt.lib()
    L.uvt_dtrmm.argtypes = [c.c_void_p, c.c_int, c.c_int, c.c_int, c.c_int, c.c_int64, c.c_int64, c.c_double,
                            c.c_void_p, c.c_int64, c.c_void_p, c.c_int64, c.c_void_p]
    m, n, ld = 67, 90, (1 << 24) + 1
    rng = np.random.default_rng(side * 8 + uplo * 4 + trans * 2 + diag)
    nt = n if side else m
    A, B = rng.integers(-2, 3, (nt, nt)).astype(np.float64), rng.integers(-2, 3, (m, n)).astype(np.float64)
    T = np.triu(A) if uplo else np.tril(A)
    if diag:
        np.fill_diagonal(T, 1.0)
    op = T.T if trans else T
    print("[gpu-long-rows] dtrmm", side, uplo, trans, diag, flush=True)
    dA, dB = strided(gpu, A, ld), strided(gpu, B, ld)
    try:
        st = L.uvt_dtrmm(gpu.ptr, side, uplo, trans, diag, m, n, 1.0, dA.ptr, ld, dB.ptr, ld, gpu.stream)
        gpu.sync()
        assert st == 0
        got = np.full((m, n), 7.5)
        dB.download_2d(got, n * 8, m, n * 8, ld * 8)
        np.testing.assert_array_equal(got, B @ op if side else op @ B)
    finally:
        dA.free()
        dB.free()
