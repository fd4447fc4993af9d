"""uvt_inf_norm on one handle from several host threads, on one stream and on a
stream each: every call gets its own matrix's norm.  (The entries are integers,
so the sums are exact.)"""
import ctypes as c
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("streams", ["one", "each"])
def test_threads_get_their_own_norm(uvt, streams):
    print("[gpu-norm]", streams, flush=True)
    gpu = uvt.Handle(0)  # its buffers are made by whichever thread comes first
    L = uvt.lib()
    rng = np.random.default_rng(3)
    shapes = [(1, 7), (40, 3000), (513, 64), (700, 900)]
    mats = [rng.integers(-9, 10, s).astype(np.float64) * (i + 1) for i, s in enumerate(shapes)]
    want = [np.abs(x).sum(axis=1).max() for x in mats]
    bufs = [gpu.array(x) for x in mats]
    own = []
    for _ in mats:
        s = c.c_void_p()
        assert L.uvt_stream_create(gpu.ptr, c.byref(s)) == 0
        own.append(s)
    wrong, start = [], threading.Barrier(len(mats))

    def work(i):
        stream = own[i] if streams == "each" else gpu.stream
        out = c.c_double()
        start.wait()
        for _ in range(300):
            st = L.uvt_inf_norm(gpu.ptr, *shapes[i], bufs[i].ptr, shapes[i][1], c.byref(out), stream)
            if st != 0 or out.value != want[i]:
                wrong.append((i, st, out.value))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(mats))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s in own:
        L.uvt_stream_destroy(gpu.ptr, s)
    for b in bufs:
        b.free()
    gpu.close()
    assert not wrong, wrong[:5]
