"""The work that is timed: calls of the TRMM engine as its users make them.

Every case is one pass through a public entry point on operands that are
already on the GPU (torch tensors here; the engine takes their addresses, and
its work goes to torch's stream), with the plan, handle, workspace, graph or
server that a program keeps between calls.  Kinds:

  trmm   C = tril(A) B in FP64 through a band plan: orders 64 .. 32768, B
         16 .. 8192 columns wide, both mappings, both shapes, padded and odd
         leading dimensions; with norm=True the infinity norm of C after it,
         which is what the command line computes.
  split  the same product in split precision (12 .. 14 moduli), orders
         512 .. 32768; with statement=True the call's error statement too.
  dgemm  C = alpha op(A) op(B) + beta C, the box call of the BLAS forms.
  dtrmm  B = alpha op(A) B or alpha B op(A) in place, the triangle call, every
         side, triangle, transpose and diagonal.
  batch  many uneven products in one graph launch.
  serve  a burst of requests submitted to the server and drained.
"""
import ctypes
import math
import os

import numpy as np
import torch

import uvatrmm_amd as uvt
from uvatrmm_amd import workloads

F64 = torch.float64
DEV = "cuda"
_HANDLE = None


def listed():
    return [
        # the smallest reference order: one call is launches and one short chain of k panels
        dict(name="trmm_257", kind="trmm", n=257, m=257, p=1, mapping="reg", shape="trapezoid",
             pad=0, spread=False, norm=False),
        # the reference's documented run, uvatrmm.x 2048 reg boxes on 4 ranks, product and norm
        dict(name="program_2048_boxes", kind="trmm", n=2048, m=2048, p=4, mapping="reg",
             shape="boxes", pad=0, spread=False, norm=True),
        # an ordinary square product
        dict(name="trmm_4096", kind="trmm", n=4096, m=4096, p=16, mapping="balanced",
             shape="trapezoid", pad=0, spread=True, norm=False),
        # narrow B: the share of one of many ranks, few and deep tiles
        dict(name="trmm_9000x250", kind="trmm", n=9000, m=250, p=8, mapping="balanced",
             shape="trapezoid", pad=0, spread=True, norm=False),
        # ragged: odd order, odd width, odd leading dimensions
        dict(name="trmm_8165x939_odd", kind="trmm", n=8165, m=939, p=16, mapping="balanced",
             shape="trapezoid", pad=0, spread=True, norm=False),
        # the headline: the largest configuration of the benchmark
        dict(name="trmm_32768x8192", kind="trmm", n=32768, m=8192, p=16, mapping="balanced",
             shape="trapezoid", pad=0, spread=True, norm=False),
        # split precision at an ordinary ragged size, default accuracy, with its error statement
        dict(name="split_5000x1500", kind="split", n=5000, m=1500, slices=13, pad=0, spread=True,
             statement=True),
        # split precision on the headline's inputs, the benchmark's 12 moduli
        dict(name="split_32768x8192", kind="split", n=32768, m=8192, slices=12, pad=0, spread=True,
             statement=False),
        # a trailing update of a blocked factorisation: C = beta C + alpha A^T B, ragged
        dict(name="dgemm_tn_update", kind="dgemm", ta=True, tb=False, m=1500, n=2000, k=3000,
             alpha=-0.5, beta=0.5, pad=0, spread=False),
        # B = B op(A) with the other triangle, transposed, unit diagonal
        dict(name="dtrmm_right_upper_t", kind="dtrmm", right=True, upper=True, trans=True,
             unit=True, m=3000, n=2048, alpha=1.0, pad=0, spread=False),
        # the benchmark's batch: 512 uneven problems, half of them split class, one graph
        dict(name="batch_512", kind="batch", count=512, sizes_seed=7, nmin=64, nmax=4096, mmin=16,
             mmax=1024, slices=12, spread=True),
        # a burst at the server: mixed sizes and tolerance classes, as many as fit the slots at once
        dict(name="serve_burst_48", kind="serve", count=48, sizes_seed=7, nmin=128, nmax=8192,
             mmin=64, mmax=2048, slices=12, slots=8, spread=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trmm"] * 8 + ["split"] * 3 + ["dgemm"] * 2 + ["dtrmm"] * 3 + ["batch", "serve"])
    pad = rng.choice([0, 0, 0, 1, 8])
    spread = rng.random() < 0.7
    if kind == "trmm":
        n = _log_int(rng, 64, 32768)
        return dict(kind=kind, n=n, m=_log_int(rng, 16, 8192), p=rng.randint(1, 16),
                    mapping=rng.choice(["reg", "balanced"]), shape=rng.choice(["trapezoid", "trapezoid", "boxes"]),
                    pad=pad, spread=spread, norm=rng.random() < 0.2)
    if kind == "split":
        return dict(kind=kind, n=_log_int(rng, 512, 32768), m=_log_int(rng, 64, 8192),
                    slices=rng.choice([12, 13, 14]), pad=pad, spread=spread, statement=rng.random() < 0.3)
    if kind == "dgemm":
        plain = rng.random() < 0.5
        return dict(kind=kind, ta=rng.random() < 0.4, tb=rng.random() < 0.4, m=_log_int(rng, 64, 8192),
                    n=_log_int(rng, 16, 8192), k=_log_int(rng, 64, 8192),
                    alpha=1.0 if plain else rng.choice([-1.0, 0.75]), beta=0.0 if plain else rng.choice([0.0, 0.5]),
                    pad=pad, spread=spread)
    if kind == "dtrmm":
        return dict(kind=kind, right=rng.random() < 0.4, upper=rng.random() < 0.4, trans=rng.random() < 0.4,
                    unit=rng.random() < 0.3, m=_log_int(rng, 64, 8192), n=_log_int(rng, 64, 8192),
                    alpha=rng.choice([1.0, 1.0, -0.75]), pad=pad, spread=spread)
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(16, 256), sizes_seed=rng.randint(0, 10**6), nmin=64,
                    nmax=rng.choice([512, 2048, 4096]), mmin=16, mmax=rng.choice([128, 1024]),
                    slices=rng.choice([12, 13]), spread=spread)
    return dict(kind=kind, count=rng.randint(4, 40), sizes_seed=rng.randint(0, 10**6), nmin=128,
                nmax=rng.choice([1024, 4096, 8192]), mmin=64, mmax=rng.choice([512, 2048]), slices=rng.choice([12, 13]),
                slots=rng.choice([4, 8]), spread=spread)


# ---------------------------------------------------------------- operands

class _Buf:
    """A torch tensor as the engine's bindings take buffers: an address and a size."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


def _handle():
    """One handle per process; its work goes to torch's stream."""
    global _HANDLE
    if _HANDLE is None:
        _HANDLE = uvt.Handle(torch.cuda.current_device())
        _HANDLE.stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    return _HANDLE


def _fill(x, g, spread):
    """U[-1, 1), with spread times 2^e, e uniform in -8 .. 8, a block of rows at a time."""
    x.uniform_(-1.0, 1.0, generator=g)
    if spread:
        rows = max(1, (1 << 27) // max(1, x.shape[-1]))
        for r in range(0, x.shape[0], rows):
            part = x[r:r + rows]
            e = torch.randint(-8, 9, part.shape, generator=g, device=DEV, dtype=torch.int32)
            part.copy_(torch.ldexp(part, e))
    return x


def _triangle(n, ld, g, spread):
    """A square matrix with a heavier diagonal; the triangle that is not used
    holds other values, as the storage of a factorisation does."""
    a = _fill(torch.empty(n, ld, dtype=F64, device=DEV), g, spread)
    a.diagonal()[:n].add_(2.0)
    return a


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _sizes(case):
    if case["kind"] == "batch":
        return workloads.batch_problems(case["sizes_seed"], case["count"], case["nmin"], case["nmax"],
                                        case["mmin"], case["mmax"])
    return workloads.serve_sizes(np.random.default_rng(case["sizes_seed"]), case["count"], case["nmin"],
                                 case["nmax"], case["mmin"], case["mmax"])


def _inputs(case, seed):
    g, kind = _gen(seed), case["kind"]
    pad, spread = case.get("pad", 0), case["spread"]
    if kind in ("trmm", "split"):
        n, m = case["n"], case["m"]
        return dict(A=_triangle(n, n + pad, g, spread),
                    B=_fill(torch.empty(n, m + pad, dtype=F64, device=DEV), g, spread))
    if kind == "dgemm":
        m, n, k = case["m"], case["n"], case["k"]
        ar, ac = (k, m) if case["ta"] else (m, k)
        br, bc = (n, k) if case["tb"] else (k, n)
        return dict(A=_fill(torch.empty(ar, ac + pad, dtype=F64, device=DEV), g, spread),
                    B=_fill(torch.empty(br, bc + pad, dtype=F64, device=DEV), g, spread),
                    C=_fill(torch.empty(m, n + pad, dtype=F64, device=DEV), g, False))
    if kind == "dtrmm":
        k = case["n"] if case["right"] else case["m"]
        return dict(A=_triangle(k, k + pad, g, spread),
                    B=_fill(torch.empty(case["m"], case["n"] + pad, dtype=F64, device=DEV), g, spread))
    # batch, serve: every operand in one pool each, at even element offsets
    # (the batch with even leading dimensions, as the benchmark lays it out;
    # the server's requests are contiguous)
    step = 2 if kind == "batch" else 1
    probs, na, nb, nc = [], 0, 0, 0
    for n, m, prec in _sizes(case):
        lda, ldb = -(-n // step) * step, -(-m // step) * step
        probs.append((n, m, prec, lda, ldb, na, nb, nc))
        na += n * lda + (n * lda & 1)
        nb += n * ldb + (n * ldb & 1)
        nc += n * m + (n * m & 1)
    A = _fill(torch.empty(na, 1, dtype=F64, device=DEV), g, spread).view(-1)
    B = _fill(torch.empty(nb, 1, dtype=F64, device=DEV), g, spread).view(-1)
    for n, m, prec, lda, ldb, oa, ob, oc in probs:
        A[oa:oa + n * lda].view(n, lda).diagonal()[:n].add_(2.0)
    return dict(A=A, B=B, C=torch.zeros(nc, dtype=F64, device=DEV), probs=probs)


# ---------------------------------------------------------------- one pass

class _Trmm:
    def __init__(self, case, seed):
        self.case, self.h = case, _handle()
        x = _inputs(case, seed)
        n, m = case["n"], case["m"]
        self.A, self.B = _Buf(x["A"]), _Buf(x["B"])
        self.C = torch.empty(n, m, dtype=F64, device=DEV)
        self.c = _Buf(self.C)
        # a mapping that leaves a band without rows is refused: such a caller takes fewer bands
        p = min(case["p"], n)
        while True:
            try:
                self.plan = uvt.Plan(n, m, p, case["mapping"], case["shape"])
                break
            except uvt.UvtError:
                if p == 1:
                    raise
                p -= 1

    def run(self):
        n, m, pad = self.case["n"], self.case["m"], self.case["pad"]
        self.h.trmm_f64(self.plan, self.A, n + pad, self.B, m + pad, self.c, m)
        if self.case["norm"]:
            return {"C": self.C, "norm": self.h.inf_norm(n, m, self.c, m)}
        return {"C": self.C}


class _Split:
    def __init__(self, case, seed):
        self.case, self.h = case, _handle()
        x = _inputs(case, seed)
        n, m = case["n"], case["m"]
        self.A, self.B = _Buf(x["A"]), _Buf(x["B"])
        self.C = torch.empty(n, m, dtype=F64, device=DEV)
        self.c = _Buf(self.C)
        self.work = _Buf(torch.empty(self.h.split_workspace(n, m, case["slices"]), dtype=torch.uint8, device=DEV))

    def run(self):
        c = self.case
        n, m, s, pad = c["n"], c["m"], c["slices"], c["pad"]
        self.h.trmm_split(n, m, s, self.A, n + pad, self.B, m + pad, self.c, m, self.work)
        if c["statement"]:
            bound, estimate = self.h.split_error(n, m, s, self.work)
            return {"C": self.C, "bound": bound, "estimate": estimate}
        return {"C": self.C}


def _i64(v):
    return ctypes.c_int64(v)


class _Dgemm:
    def __init__(self, case, seed):
        self.h = _handle()
        x = _inputs(case, seed)
        self.A, self.B, self.C = x["A"], x["B"], x["C"]
        self.n = case["n"]
        self.args = (self.h.ptr, int(case["ta"]), int(case["tb"]), _i64(case["m"]), _i64(case["n"]), _i64(case["k"]),
                     ctypes.c_double(case["alpha"]), ctypes.c_void_p(self.A.data_ptr()), _i64(self.A.shape[1]),
                     ctypes.c_void_p(self.B.data_ptr()), _i64(self.B.shape[1]), ctypes.c_double(case["beta"]),
                     ctypes.c_void_p(self.C.data_ptr()), _i64(self.C.shape[1]), self.h.stream)

    def run(self):
        uvt.check(uvt.lib().uvt_dgemm(*self.args), "dgemm")
        return {"C": self.C[:, :self.n]}


class _Dtrmm:
    """The call overwrites B, so the pass starts from the caller's B again."""

    def __init__(self, case, seed):
        self.h = _handle()
        x = _inputs(case, seed)
        self.A, self.B0 = x["A"], x["B"]
        self.B = torch.empty_like(self.B0)
        self.n = case["n"]
        self.args = (self.h.ptr, int(case["right"]), int(case["upper"]), int(case["trans"]), int(case["unit"]),
                     _i64(case["m"]), _i64(case["n"]), ctypes.c_double(case["alpha"]),
                     ctypes.c_void_p(self.A.data_ptr()), _i64(self.A.shape[1]),
                     ctypes.c_void_p(self.B.data_ptr()), _i64(self.B.shape[1]), self.h.stream)

    def run(self):
        self.B.copy_(self.B0)
        uvt.check(uvt.lib().uvt_dtrmm(*self.args), "dtrmm")
        return {"B": self.B[:, :self.n]}


class _Batch:
    def __init__(self, case, seed):
        self.h = _handle()
        x = _inputs(case, seed)
        self.x, self.C = x, x["C"]
        a, b, c = (x[k].data_ptr() for k in "ABC")
        self.batch = uvt.Batch(self.h, [uvt.Problem(a + 8 * oa, lda, b + 8 * ob, ldb, c + 8 * oc, m, n, m, prec,
                                                    uvt.ROUTE_AUTO)
                                        for n, m, prec, lda, ldb, oa, ob, oc in x["probs"]], slices=case["slices"],
                               table=os.path.join(uvt.HERE, "tune", "f64_tiles.json"))

    def run(self):
        self.batch.run()
        return {"C": self.C}

    def __del__(self):
        if hasattr(self, "batch"):
            self.batch.close()


class _Serve:
    def __init__(self, case, seed):
        self.h = _handle()
        x = _inputs(case, seed)
        self.x, self.C = x, x["C"]
        a, b, c = (x[k].data_ptr() for k in "ABC")
        self.server = uvt.Server(self.h, 8 << 30, max_slots=case["slots"], slices=case["slices"])
        self.reqs = []
        for n, m, prec, lda, ldb, oa, ob, oc in x["probs"]:
            bufs = []
            for base, off in ((a, oa), (b, ob), (c, oc)):
                v = _Buf.__new__(_Buf)
                v.t, v.ptr, v.nbytes = None, base + 8 * off, 0
                bufs.append(v)
            self.reqs.append((n, m, prec, *bufs))

    def run(self):
        for n, m, prec, a, b, c in self.reqs:
            self.server.submit_device(n, m, prec, a, b, c)
        self.server.drain()
        for done in self.server.poll():
            uvt.check(done["status"], "request")
        return {"C": self.C}

    def __del__(self):
        if hasattr(self, "server"):
            self.server.close()


_KINDS = dict(trmm=_Trmm, split=_Split, dgemm=_Dgemm, dtrmm=_Dtrmm, batch=_Batch, serve=_Serve)


def prepare(case, seed):
    return _KINDS[case["kind"]](case, seed)


def run(state):
    return state.run()


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind in ("trmm", "split"):
        n, m = case["n"], case["m"]
        return {"bytes": 8.0 * (n * (n + 1) / 2 + 2.0 * n * m), "flops": float(m) * n * n}
    if kind == "dgemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 8.0 * (m * k + k * n + m * n * (2 if case["beta"] else 1)), "flops": 2.0 * m * n * k}
    if kind == "dtrmm":
        m, n = case["m"], case["n"]
        k, w = (n, m) if case["right"] else (m, n)
        return {"bytes": 8.0 * (k * (k + 1) / 2 + 2.0 * k * w), "flops": float(w) * k * k}
    by = fl = 0.0
    for n, m, _ in _sizes(case):
        by += 8.0 * (n * (n + 1) / 2 + 2.0 * n * m)
        fl += float(m) * n * n
    return {"bytes": by, "flops": fl}


# ---------------------------------------------------------------- the same results from plain torch

def exact(case, seed):
    x, kind = _inputs(case, seed), case["kind"]
    if kind in ("trmm", "split"):
        n, m = case["n"], case["m"]
        c = torch.tril(x["A"][:, :n]) @ x["B"][:, :m].contiguous()
        if kind == "trmm":
            return {"C": c, "norm": float(c.abs().sum(1).max())} if case["norm"] else {"C": c}
        return {"C": c, "bound": None, "estimate": None} if case["statement"] else {"C": c}
    if kind == "dgemm":
        m, n, k = case["m"], case["n"], case["k"]
        a = x["A"][:, :m].t() if case["ta"] else x["A"][:, :k]
        b = x["B"][:, :k].t() if case["tb"] else x["B"][:, :n]
        return {"C": case["alpha"] * (a.contiguous() @ b.contiguous()) + case["beta"] * x["C"][:, :n]}
    if kind == "dtrmm":
        k = x["A"].shape[0]
        a = x["A"][:, :k]
        t = torch.triu(a) if case["upper"] else torch.tril(a)
        if case["unit"]:
            t.diagonal().fill_(1.0)
        t = (t.t() if case["trans"] else t).contiguous()
        b = x["B"][:, :case["n"]].contiguous()
        return {"B": case["alpha"] * (b @ t if case["right"] else t @ b)}
    A, B, C = x["A"], x["B"], x["C"]
    for n, m, _, lda, ldb, oa, ob, oc in x["probs"]:
        a = torch.tril(A[oa:oa + n * lda].view(n, lda)[:, :n])
        C[oc:oc + n * m] = (a @ B[ob:ob + n * ldb].view(n, ldb)[:, :m].contiguous()).view(-1)
    return {"C": C}
