"""uvt_batch_update on the MI355X and the alignment of operands: other leading
dimensions and addresses of the same alignment are taken, others refused with
UVT_ERR_ARG, which leaves the batch as it was."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("odd", [0, 1])
def test_alignment_is_kept(uvt, gpu, odd):
    n, m = 130, 67 + odd
    rng = np.random.default_rng(odd)
    A = np.tril(rng.integers(-3, 4, (n, n))).astype(np.float64)
    B = rng.integers(-3, 4, (n, m)).astype(np.float64)

    def place(pad_a, pad_b, shift):
        Ap, Bp = np.full((n, n + pad_a), np.nan), np.full(n * (m + pad_b) + 1, np.nan)
        Ap[:, :n] = A
        Bp[shift:shift + n * (m + pad_b)].reshape(n, m + pad_b)[:, :m] = B
        dA, dB, dC = gpu.array(Ap), gpu.array(Bp), gpu.array(np.full((n, m), np.nan))
        bufs.extend((dA, dB, dC))
        return dC, uvt.Problem(dA.ptr, n + pad_a, dB.ptr + 8 * shift, m + pad_b, dC.ptr, m, n, m, uvt.PREC_F64, 0)

    bufs = []
    print("[gpu-batch-update]", odd, flush=True)
    # even: lda 130 and ldb even; odd: ldb odd
    dC, prob = place(0, 1, 0)
    assert (prob.ldb % 2 == 1) == bool(odd)
    batch = uvt.Batch(gpu, [prob])
    same = [place(2, prob.ldb - m + 2, 0)] + ([place(1, 1, 0), place(0, 0, 1)] if odd else [])
    for dD, p in same:
        batch.update([p])
        batch.run()
        gpu.sync()
        np.testing.assert_array_equal(dD.download((n, m)), A @ B)
    other = [place(0, 0, 0)] if odd else [place(1, 1, 0), place(0, 2, 0), place(0, 1, 1)]
    last = same[-1][0]
    for dD, p in other:
        with pytest.raises(uvt.UvtError) as e:
            batch.update([p])
        assert e.value.status == uvt.ERR_ARG
        last.zero()
        batch.run()
        gpu.sync()
        np.testing.assert_array_equal(last.download((n, m)), A @ B)
        assert np.isnan(dD.download((n, m))).all()
    batch.close()
    for b in bufs:
        b.free()
