"""uvt_dgemm on the MI355X with shallow reductions, on both sides of the lines
where it changes from wave tiles to workgroup tiles and from one order of the
tiles to the other, with C written and with C updated.  Small integers and
power-of-two factors make every sum exact, so results equal NumPy's bit for
bit; NaN surrounds the operands."""
import ctypes as c

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def padded(x, pad, fill=np.nan):
    y = np.full((x.shape[0], x.shape[1] + pad), fill)
    y[:, :x.shape[1]] = x
    return y


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("m,n,k", [(767, 768, 64), (769, 768, 64), (769, 768, 65), (1031, 1100, 1), (1031, 1100, 16),
                                   (4096, 4090, 32), (4097, 4090, 17), (4097, 4090, 33), (130, 40001, 31)])
def test_dgemm_shallow_exact(uvt, gpu, m, n, k, ta, tb):
    L = uvt.lib()
    L.uvt_dgemm.argtypes = [c.c_void_p, c.c_int, c.c_int, c.c_int64, c.c_int64, c.c_int64, c.c_double, c.c_void_p,
                            c.c_int64, c.c_void_p, c.c_int64, c.c_double, c.c_void_p, c.c_int64, c.c_void_p]
    rng = np.random.default_rng(m + k)
    A = rng.integers(-3, 4, (k, m) if ta else (m, k)).astype(np.float64)
    B = rng.integers(-3, 4, (n, k) if tb else (k, n)).astype(np.float64)
    C = rng.integers(-3, 4, (m, n)).astype(np.float64)
    prod = (A.T if ta else A) @ (B.T if tb else B)
    for alpha, beta in ((1.0, 0.0), (-2.0, 0.0), (-2.0, 0.5)):
        print("[gpu-shallow]", (m, n, k), (ta, tb), alpha, beta, flush=True)
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
