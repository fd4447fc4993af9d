"""uvt_dgemm and uvt_dtrmm on the MI355X with operands that share memory: the
result is that of the inputs as they were before the call.  Small integers and
power-of-two factors make every sum exact, so results equal NumPy's bit for
bit, at sizes of one wave tile, of many wave tiles and of workgroup tiles."""
import ctypes as c
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [5, 130, 1400]


@pytest.fixture(scope="module")
def L(uvt, gpu):
    lib = uvt.lib()
    args = [c.c_void_p, c.c_int, c.c_int, c.c_int, c.c_int, c.c_int64, c.c_int64, c.c_double, c.c_void_p, c.c_int64,
            c.c_void_p, c.c_int64, c.c_void_p]
    lib.uvt_dtrmm.argtypes = lib.uvt_dtrmm_noalloc.argtypes = args
    lib.uvt_dgemm.argtypes = [c.c_void_p, c.c_int, c.c_int, c.c_int64, c.c_int64, c.c_int64, c.c_double, c.c_void_p,
                              c.c_int64, c.c_void_p, c.c_int64, c.c_double, c.c_void_p, c.c_int64, c.c_void_p]
    return lib


def ints(rng, *shape):
    return rng.integers(-2, 3, shape).astype(np.float64)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("which", ["A", "B", "shifted"])
@pytest.mark.parametrize("ta,tb,alpha,beta", [(0, 0, -2.0, 0.5), (0, 0, 1.0, 0.0), (1, 0, 1.0, 0.0), (0, 1, 1.0, 0.5),
                                              (1, 1, -1.0, 0.0)])
def test_dgemm_result_over_an_operand(L, gpu, n, which, ta, tb, alpha, beta):
    rng = np.random.default_rng(n)
    ld, off = n + 3, 2 * (n + 3) + 1  # shifted: C starts inside A
    mem, B = ints(rng, n + 2, ld), ints(rng, n, n)
    A = mem[:n, :n].copy()
    dM, dB = gpu.array(mem), gpu.array(B)
    Cp, ldc = dM.ptr, ld
    C = A
    if which == "B":
        Cp, ldc, C = dB.ptr, n, B
    if which == "shifted":
        Cp, C = dM.ptr + 8 * off, mem[2:n + 2, 1:n + 1].copy()
    want = alpha * ((A.T if ta else A) @ (B.T if tb else B)) + (beta * C if beta else 0.0)
    print("[gpu-overlap] dgemm", n, which, ta, tb, alpha, beta, flush=True)
    st = L.uvt_dgemm(gpu.ptr, ta, tb, n, n, n, alpha, dM.ptr, ld, dB.ptr, n, beta, Cp, ldc, gpu.stream)
    gpu.sync()
    M, Bn = dM.download(mem.shape), dB.download((n, n))
    dM.free()
    dB.free()
    assert st == 0
    got = Bn if which == "B" else M[:n, :n] if which == "A" else M[2:n + 2, 1:n + 1]
    np.testing.assert_array_equal(got, want)
    same = np.ones(mem.shape, bool)  # nothing else is written
    if which != "B":
        same[2:n + 2, 1:n + 1] = which == "A"
        same[:n, :n] &= which != "A"
    np.testing.assert_array_equal(M[same], mem[same])


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("noalloc", [0, 1])
@pytest.mark.parametrize("side,uplo,trans,diag", list(itertools.product((0, 1), repeat=4)))
def test_dtrmm_over_its_own_triangle(L, gpu, n, noalloc, side, uplo, trans, diag):
    """B is the memory of A's square."""
    rng = np.random.default_rng(n + 1)
    M = ints(rng, n, n + 1)
    T = np.triu(M[:, :n]) if uplo else np.tril(M[:, :n])
    if diag:
        np.fill_diagonal(T, 1.0)
    op, B = (T.T if trans else T), M[:, :n]
    want = -2.0 * (B @ op if side else op @ B)
    dM = gpu.array(M)
    print("[gpu-overlap] dtrmm", n, noalloc, side, uplo, trans, diag, flush=True)
    f = L.uvt_dtrmm_noalloc if noalloc else L.uvt_dtrmm
    st = f(gpu.ptr, side, uplo, trans, diag, n, n, -2.0, dM.ptr, n + 1, dM.ptr, n + 1, gpu.stream)
    gpu.sync()
    got = dM.download(M.shape)
    dM.free()
    assert st == 0
    np.testing.assert_array_equal(got[:, :n], want)
    np.testing.assert_array_equal(got[:, n], M[:, n])


@pytest.mark.parametrize("n", SIZES[1:])
def test_dtrmm_in_the_unused_triangle(L, gpu, n):
    """B is a block above the diagonal of the square that holds A."""
    rng = np.random.default_rng(n + 2)
    M = ints(rng, 2 * n, 2 * n)
    T = np.tril(M)[:n, :n]
    want = M.copy()
    want[:n, n:] = T @ M[:n, n:]
    dM = gpu.array(M)
    print("[gpu-overlap] block", n, flush=True)
    st = L.uvt_dtrmm(gpu.ptr, 0, 0, 0, 0, n, n, 1.0, dM.ptr, 2 * n, dM.ptr + 8 * n, 2 * n, gpu.stream)
    gpu.sync()
    got = dM.download(M.shape)
    dM.free()
    assert st == 0
    np.testing.assert_array_equal(got, want)
