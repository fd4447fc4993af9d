"""The batch kernel's queues, one per XCD: batches with fewer tiles than
queues, with one problem only (most workgroups draw from other queues than
their own), with more tiles than resident workgroups, and with one deep
problem among many small ones.  Every tile is run once, so each result
matches the FP64 oracle, and replays give the same bits."""
import numpy as np
import pytest

from conftest import rel_fro

pytestmark = pytest.mark.gpu

CASES = {
    "one tile": [(5, 3)],
    "seven tiles": [(40 + k, 17) for k in range(7)],
    "nine tiles": [(64, 20 + k) for k in range(9)],
    "one problem": [(1100, 1130)],
    "two row blocks": [(200, 1000)],
    "1200 one-tile problems": [(30 + k % 34, 8 + k % 25) for k in range(1200)],
    "one deep problem": [(60 + k % 9, 33) for k in range(200)] + [(2500, 40)],
    "uneven": [(1800, 290), (130, 129), (900, 65), (257, 1), (64, 700), (1025, 128)] * 3,
}


@pytest.mark.parametrize("name", list(CASES))
def test_every_tile_runs_once(uvt, gpu, oracle, name):
    sizes = CASES[name]
    rng = np.random.default_rng(len(sizes))
    print("[gpu-batch-queues]", name, flush=True)
    probs, host, bufs = [], [], []
    for n, m in sizes:
        A, B = np.tril(rng.standard_normal((n, n))), rng.standard_normal((n, m))
        C = np.full((n, m), np.nan)
        d = gpu.array(A), gpu.array(B), gpu.array(C)
        host.append((A, B))
        bufs.append(d)
        probs.append(uvt.Problem(d[0].ptr, n, d[1].ptr, m, d[2].ptr, m, n, m, uvt.PREC_F64, 0))
    batch = uvt.Batch(gpu, probs, slices=12)
    first = None
    for _ in range(3):
        batch.run()
        gpu.sync()
        out = [b[2].download(s) for b, s in zip(bufs, sizes)]
        if first is None:
            first = out
            for (A, B), c in zip(host, out):
                assert rel_fro(c, oracle.trmm(A, B)) <= 1e-13
        else:
            for x, y in zip(first, out):
                np.testing.assert_array_equal(x, y)
    batch.close()
