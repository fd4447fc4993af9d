"""Edge tiles of the FP64 kernels on the MI355X: orders and widths around the
tile sizes, odd and even leading dimensions, with everything outside the
operands poisoned.  Small-integer inputs make every sum exact in any order, so
the results equal NumPy's bit for bit and no poison reaches C."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", ["trapezoid", "boxes"])
@pytest.mark.parametrize("n,m", [(1, 1), (15, 2), (17, 3), (63, 65), (65, 1), (129, 63), (257, 127),
                                 (130, 33), (640, 97), (641, 129), (2305, 3201)])
def test_edges_with_poisoned_surroundings(gpu, uvt, n, m, shape):
    rng = np.random.default_rng(n * 31 + m)
    A = rng.integers(-3, 4, (n, n)).astype(np.float64)
    B = rng.integers(-3, 4, (n, m)).astype(np.float64)
    want = np.tril(A) @ B
    A[np.triu_indices(n, 1)] = np.nan
    for pa, pb in ((0, 0), (1, 1), (1, 2), (4, 3)):
        Ap, Bp = np.full((n, n + pa), np.nan), np.full((n, m + pb), np.nan)
        Ap[:, :n], Bp[:, :m] = A, B
        print("[gpu-edges]", n, m, shape, pa, pb, flush=True)
        plan = uvt.Plan(n, m, min(3, n), "reg", shape)
        dA, dB, dC = gpu.array(Ap), gpu.array(Bp), gpu.array(np.full((n, m + pb), 7.5))
        gpu.trmm_f64(plan, dA, n + pa, dB, m + pb, dC, m + pb)
        gpu.sync()
        C = dC.download((n, m + pb))
        plan.close()
        for b in (dA, dB, dC):
            b.free()
        np.testing.assert_array_equal(C[:, :m], want)
        assert (C[:, m:] == 7.5).all()  # nothing written outside C
