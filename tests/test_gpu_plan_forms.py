"""Which form a plan's launch takes on the MI355X, and its results there: sizes
past the lines where wave tiles end, with odd orders, widths and leading
dimensions and NaN in everything that is not an operand.  The launch's
workgroups and partial tiles tell the form.  Small-integer inputs make every
sum exact in any order, so results equal NumPy's bit for bit."""
import ctypes as c

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def tiles(n, m, tm, tn):
    return -(-n // tm) * -(-m // tn)


def run(gpu, uvt, n, m, shape, pads):
    rng = np.random.default_rng(n * 13 + m)
    A = rng.integers(-2, 3, (n, n)).astype(np.float64)
    B = rng.integers(-2, 3, (n, m)).astype(np.float64)
    want = np.tril(A) @ B
    A[np.triu_indices(n, 1)] = np.nan
    plan = uvt.Plan(n, m, 3, "reg", shape)
    launch = gpu.plan_launch_info(plan)
    for pa, pb in pads:
        print("[gpu-plan-forms]", n, m, shape, pa, pb, launch, flush=True)
        Ap, Bp = np.full((n, n + pa), np.nan), np.full((n, m + pb), np.nan)
        Ap[:, :n], Bp[:, :m] = A, B
        dA, dB, dC = gpu.array(Ap), gpu.array(Bp), gpu.array(np.full((n, m + pb), 7.5))
        gpu.trmm_f64(plan, dA, n + pa, dB, m + pb, dC, m + pb)
        gpu.sync()
        C = dC.download((n, m + pb))
        for b in (dA, dB, dC):
            b.free()
        np.testing.assert_array_equal(C[:, :m], want)
        assert (C[:, m:] == 7.5).all()
    plan.close()
    return launch


def waves(n, m, tm, tn):
    """Workgroups of four one-wave tiles, two along the columns where there are
    two."""
    rt, ct = -(-n // tm), -(-m // tn)
    wn = 2 if ct > 1 else 1
    return -(-rt // (4 // wn)) * -(-ct // wn)


@pytest.mark.parametrize("n,m,shape,form,tm,tn", [
    (1023, 31, "boxes", "waves", 16, 16),
    (1023, 701, "trapezoid", "waves", 16, 32),
    (1301, 2003, "boxes", "waves", 32, 32),
    (769, 4001, "trapezoid", "waves", 32, 32),
    (2049, 1999, "boxes", "tiles", 64, 64),
    (2177, 2111, "trapezoid", "tiles", 64, 64),
    (5001, 301, "boxes", "cut", 64, 64),
    (9001, 33, "trapezoid", "cut", 128, 32),
    (1301, 8001, "boxes", "tiles", 128, 128),
    (5001, 1711, "boxes", "stream-k", 128, 128),
])
def test_each_form_with_poisoned_surroundings(gpu, uvt, n, m, shape, form, tm, tn):
    wg, parts = run(gpu, uvt, n, m, shape, ((0, 0), (1, 1), (2, 3)) if n < 4000 else ((1, 1),))
    if form == "waves":
        assert (wg, parts) == (waves(n, m, tm, tn), 0)
    elif form == "tiles":
        assert (wg, parts) == (tiles(n, m, tm, tn), 0)
    elif form == "cut":
        assert parts > 0 and wg == tiles(n, m, tm, tn) + parts
    else:
        assert parts > 0 and wg <= 2 * gpu.cus and wg > 2 * gpu.cus - tiles(1, m, tm, tn)


def test_whole_narrow_tiles(gpu, uvt):
    """128x32 tiles are run whole only past n = 32768 and under 2e9 flops: a
    triangle of 8.7 GB, zero but for some rows, with NaN above their diagonal."""
    n, m, ld = 33001, 1, 33003
    rng = np.random.default_rng(9)
    rows = np.unique(np.concatenate([[0, 1, 15, 16, 127, 128, 129, n - 129, n - 2, n - 1], rng.integers(0, n, 60)]))
    B = rng.integers(-2, 3, (n, m)).astype(np.float64)
    want = np.zeros((n, m))
    dA, dB, dC = gpu.alloc(n * ld * 8), gpu.array(B), gpu.array(np.full((n, m), np.nan))
    dA.zero()
    L = uvt.lib()
    for r in rows:
        a = np.full(ld, np.nan)
        a[:r + 1] = rng.integers(-2, 3, r + 1)
        want[r] = a[:r + 1] @ B[:r + 1]
        assert L.uvt_memcpy(gpu.ptr, dA.ptr + int(r) * ld * 8, a.ctypes.data, ld * 8, 0) == 0
    plan = uvt.Plan(n, m)
    print("[gpu-plan-forms]", n, m, gpu.plan_launch_info(plan), flush=True)
    assert gpu.plan_launch_info(plan) == (tiles(n, m, 128, 32), 0)
    gpu.trmm_f64(plan, dA, ld, dB, m, dC, m)
    gpu.sync()
    got = dC.download((n, m))
    plan.close()
    for b in (dA, dB, dC):
        b.free()
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("n,m", [(7000, 19), (7001, 41), (9000, 31), (7003, 101), (27000, 3)])
def test_deep_narrow_plans_cut_their_reductions(gpu, uvt, n, m):
    """From n = 7000 to 27000, of 2e9 flops or more (m > 40 at n = 7000): else
    waves."""
    tm, tn = (128, 32) if m <= 48 else (64, 64)
    wg, parts = run(gpu, uvt, n, m, "trapezoid", ((1, 1),))
    if float(m) * n * n < 2e9 or n >= 27000:
        assert parts == 0
    else:
        assert parts > 0 and wg == tiles(n, m, tm, tn) + parts


def test_deep_plan_first_used_in_a_capture(gpu, uvt):
    """A plan that has no records on the device yet can be captured (in wave
    tiles, which need none); every replay gives the product, with eager calls of
    the plan, which cut, in between."""
    n, m = 7111, 45
    rng = np.random.default_rng(5)
    A = rng.integers(-2, 3, (n, n)).astype(np.float64)
    B = rng.integers(-2, 3, (n, m)).astype(np.float64)
    want = np.tril(A) @ B
    hip = c.CDLL(next(x.split()[-1] for x in open("/proc/self/maps") if "libamdhip64" in x))
    dA, dB, dC = gpu.array(A), gpu.array(B), gpu.alloc(n * m * 8)
    plan = uvt.Plan(n, m)
    graph, ex = c.c_void_p(), c.c_void_p()
    print("[gpu-plan-forms] capture", n, m, flush=True)
    assert hip.hipStreamBeginCapture(gpu.stream, 1) == 0  # thread-local
    gpu.trmm_f64(plan, dA, n, dB, m, dC, m)
    assert hip.hipStreamEndCapture(gpu.stream, c.byref(graph)) == 0
    assert hip.hipGraphInstantiate(c.byref(ex), graph, None, None, c.c_size_t(0)) == 0
    for _ in range(3):
        dC.zero()
        assert hip.hipGraphLaunch(ex, gpu.stream) == 0
        gpu.sync()
        np.testing.assert_array_equal(dC.download((n, m)), want)
        dC.zero()
        gpu.trmm_f64(plan, dA, n, dB, m, dC, m)
        gpu.sync()
        np.testing.assert_array_equal(dC.download((n, m)), want)
    hip.hipGraphExecDestroy(ex)
    hip.hipGraphDestroy(graph)
    plan.close()
    for b in (dA, dB, dC):
        b.free()
