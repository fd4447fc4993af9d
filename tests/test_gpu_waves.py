"""FP64 products in wave tiles on the MI355X (one wave per 16x16, 16x32 or 32x32
tile of C): sizes around the tile edges and on both sides of the lines where
the shape changes, odd leading dimensions, NaN in everything that is not an
operand, both plan shapes.  Small-integer inputs make every sum exact in any
order, so results equal NumPy's bit for bit; on seeded inputs the bits are
those of the workgroup tiles, which the batch runs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (15, 17), (16, 16), (17, 33), (31, 1), (33, 31), (257, 16), (64, 8192),  # 16x16
         (400, 1616), (300, 3001), (1023, 700), (511, 4001),                              # 16x32
         (1100, 1777), (513, 6401), (2001, 1301)]                                         # 32x32


@pytest.mark.parametrize("n,m", SIZES)
def test_exact_with_poisoned_surroundings(gpu, uvt, n, m):
    rng = np.random.default_rng(n * 17 + m)
    A = rng.integers(-3, 4, (n, n)).astype(np.float64)
    B = rng.integers(-3, 4, (n, m)).astype(np.float64)
    want = np.tril(A) @ B
    A[np.triu_indices(n, 1)] = np.nan
    for pa, pb, shape in ((0, 0, "trapezoid"), (1, 1, "boxes"), (2, 3, "trapezoid")):
        Ap, Bp = np.full((n, n + pa), np.nan), np.full((n, m + pb), np.nan)
        Ap[:, :n], Bp[:, :m] = A, B
        print("[gpu-waves]", n, m, pa, pb, shape, flush=True)
        plan = uvt.Plan(n, m, 1, "reg", shape)
        wg, parts = gpu.plan_launch_info(plan)
        assert wg > 0 and parts == 0
        dA, dB, dC = gpu.array(Ap), gpu.array(Bp), gpu.array(np.full((n, m + pb), 7.5))
        gpu.trmm_f64(plan, dA, n + pa, dB, m + pb, dC, m + pb)
        gpu.sync()
        C = dC.download((n, m + pb))
        plan.close()
        for b in (dA, dB, dC):
            b.free()
        np.testing.assert_array_equal(C[:, :m], want)
        assert (C[:, m:] == 7.5).all()


@pytest.mark.parametrize("n,m", [(259, 130), (1100, 400), (1300, 1701)])
def test_same_bits_as_workgroup_tiles(gpu, uvt, oracle, n, m):
    A, B = oracle.seeded_A(n, 3, 1), oracle.seeded_B(n, m, 3, 1)
    print("[gpu-waves] bits", n, m, flush=True)
    dA, dB, dC, dD = gpu.array(A), gpu.array(B), gpu.alloc(n * m * 8), gpu.alloc(n * m * 8)
    plan = uvt.Plan(n, m)
    gpu.trmm_f64(plan, dA, n, dB, m, dC, m)
    batch = uvt.Batch(gpu, [uvt.Problem(dA.ptr, n, dB.ptr, m, dD.ptr, m, n, m, uvt.PREC_F64, 0)])
    batch.run()
    gpu.sync()
    np.testing.assert_array_equal(dC.download((n, m)), dD.download((n, m)))
    batch.close()
    plan.close()
    for b in (dA, dB, dC, dD):
        b.free()
