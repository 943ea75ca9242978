"""Performance cases: what programs have this library do, through the entry points they call.

A case is a dict of plain values.  Kinds:
  dgemm, zgemm   one oz2.Ozaki2.gemm / zgemm call on device buffers (column-major, padded leading
                 dimensions where `pad` is set), the handle kept from call to call
  noalloc        the same DGEMM through gemm_noalloc (fixed scratch, for serving loops)
  batch          a plan of `count` uneven DGEMMs with moduli from the learned selector, replayed as a
                 graph; `reselect` chooses the moduli again from the current contents before each run
Entries: "unit" U[-1, 1); "wide" (1 + U[0, 1)) (+-1) 2^e with e uniform in [-12, 12].
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "os2-xe_amd"))
import oz2  # noqa: E402


def _gemm(name, kind, m, n, k, s, ta="N", tb="N", alpha=1.0, beta=0.0, pad=0, values="unit"):
    return dict(name=name, kind=kind, m=m, n=n, k=k, s=s, ta=ta, tb=tb, alpha=alpha, beta=beta, pad=pad, values=values)


def _batch(name, count, lo, hi, reselect, tuned, ops):
    return dict(name=name, kind="batch", count=count, lo=lo, hi=hi, reselect=reselect, tuned=tuned, ops=ops)


def listed():
    return [
        # a block of a small dense solver: the call's latency is what its caller waits for
        _gemm("dgemm_64", "dgemm", 64, 64, 64, 16),
        # the size that the CPU baseline runs, an ordinary product of a program that calls often
        _gemm("dgemm_1024", "dgemm", 1024, 1024, 1024, 14),
        # sizes as an application has them, odd leading dimensions, accumulated into C
        _gemm("dgemm_ragged", "dgemm", 1537, 771, 3001, 15, "T", "T", -1.0, 1.0, pad=3),
        # trailing update of a blocked factorisation: a short k and a large C
        _gemm("dgemm_update", "dgemm", 4096, 4096, 256, 16, "N", "T", -1.0, 1.0),
        # few moduli: the fast setting for callers that need about single precision
        _gemm("dgemm_4096_s8", "dgemm", 4096, 4096, 4096, 8, "T", "N"),
        # the headline product
        _gemm("dgemm_8192_s16", "dgemm", 8192, 8192, 8192, 16, alpha=1.5, beta=0.5),
        # a Gram-like product over a very long k with wide exponents: several k-chunks, all 24 moduli
        _gemm("dgemm_long_k", "dgemm", 2048, 2048, 200000, 24, values="wide"),
        # complex, conjugated and padded: the headline complex product
        _gemm("zgemm_4096", "zgemm", 4096, 4096, 4096, 16, "C", "N", 1.5, 0.5, pad=8),
        # complex at an ordinary odd size
        _gemm("zgemm_ragged", "zgemm", 777, 1023, 515, 16, "N", "C", pad=1),
        # a serving loop that may not allocate: C in panels through the fixed scratch
        _gemm("noalloc_1500", "noalloc", 1500, 900, 2000, 16, "N", "T"),
        # the uneven mix with the tiles and the schedule that the autotuner settles on for it
        _batch("batch_256", 256, 64, 4096, False, True, "N"),
        # a smaller mix with new contents at every run and a plan left to the defaults
        _batch("batch_64_reselect", 64, 64, 1024, True, False, "mixed"),
    ]


_MOST_OPS = 2.0 * 2048 * 2048 * 200000 * 24  # int8 operations of the largest listed case
_MOST_BYTES = 4 << 30                         # of one operand


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dgemm", "dgemm", "dgemm", "zgemm", "noalloc", "batch"])
    if kind == "batch":
        c = _batch("", _log_int(rng, 8, 256), 64, _log_int(rng, 256, 4096), rng.random() < 0.5, rng.random() < 0.5,
                   rng.choice(["N", "mixed"]))
        del c["name"]
        return c
    while True:
        hi = {"dgemm": 8192, "zgemm": 4096, "noalloc": 2048}[kind]
        m, n = _log_int(rng, 16, hi), _log_int(rng, 16, hi)
        k = _log_int(rng, 16, 4 * hi if rng.random() < 0.8 else (200000 if kind == "dgemm" else hi))
        s = rng.choice([8, 10, 12, 14, 15, 16, 16, 16, 18, 20, 22, 24])
        c = _gemm("", kind, m, n, k, s, rng.choice("NTC" if kind == "zgemm" else "NT"),
                  rng.choice("NTC" if kind == "zgemm" else "NT"), rng.choice([1.0, -1.0, 1.5]), rng.choice([0.0, 0.0, 1.0, 0.5]),
                  rng.choice([0, 0, 1, 8, 13]), rng.choice(["unit", "unit", "wide"]))
        del c["name"]
        if kind == "noalloc" and k > 8192:  # longer products do not fit the fixed scratch
            continue
        if work(c)["flops"] <= 0.5 * _MOST_OPS and 16 * max(m, n) * k <= _MOST_BYTES:
            return c


def _values(count, values, g):
    if values == "unit":
        return torch.rand(count, dtype=torch.float64, device="cuda", generator=g) * 2 - 1
    e = torch.randint(-12, 13, (count,), device="cuda", generator=g).double()
    sign = torch.randint(0, 2, (count,), device="cuda", generator=g).double() * 2 - 1
    return (1 + torch.rand(count, dtype=torch.float64, device="cuda", generator=g)) * sign * torch.exp2(e)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _gemm_inputs(case, seed):
    """(A, lda), (B, ldb), (C, ldc): flat column-major buffers of doubles, complex entries interleaved"""
    g = _generator(seed)
    m, n, k, pad = case["m"], case["n"], case["k"], case["pad"]
    width = 2 if case["kind"] == "zgemm" else 1
    out = []
    for rows, cols, values in ((m, k, case["values"]) if case["ta"] == "N" else (k, m, case["values"]),
                               (k, n, case["values"]) if case["tb"] == "N" else (n, k, case["values"]), (m, n, "unit")):
        ld = rows + pad
        out.append((_values(width * ld * cols, values, g), ld))
    return out


def _batch_problems(case, seed):
    """the problems of a batch over views of one flat C buffer; sizes from the case, contents from the seed"""
    rng = np.random.default_rng([case["count"], case["lo"], case["hi"]])
    g = _generator(seed)
    probs, total = [], 0
    for i in range(case["count"]):
        m, n, k = (int(round(math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]))))) for _ in range(3))
        ta, tb = ("NT"[rng.integers(2)], "NT"[rng.integers(2)]) if case["ops"] == "mixed" else ("N", "N")
        values = "wide" if i % 2 else "unit"
        probs.append(dict(ta=ta, tb=tb, m=m, n=n, k=k, alpha=1.0, beta=0.0, A=_values(m * k, values, g),
                          lda=m if ta == "N" else k, B=_values(k * n, values, g), ldb=k if tb == "N" else n, ldc=m))
        total += m * n
    C = torch.zeros(total, dtype=torch.float64, device="cuda")
    at = 0
    for p in probs:
        p["C"] = C[at:at + p["m"] * p["n"]]
        at += p["m"] * p["n"]
    return probs, C


def prepare(case, seed):
    oz = oz2.Ozaki2()
    if case["kind"] == "batch":
        probs, C = _batch_problems(case, seed)
        n = len(probs)
        plan = dict(tiles=[128] * n, persistent=True, largest_first=False) if case["tuned"] else {}
        b = oz2.Batch(oz, probs, bits=53, graph=True, select=True, **plan)
        return dict(oz=oz, batch=b, C=C, case=case)
    (A, lda), (B, ldb), (C, ldc) = _gemm_inputs(case, seed)
    return dict(oz=oz, A=A, lda=lda, B=B, ldb=ldb, C=C, ldc=ldc, case=case)


def run(state):
    c = state["case"]
    if c["kind"] == "batch":
        if c["reselect"]:
            state["batch"].reselect()
        state["batch"].run()
        return state["C"]
    oz = state["oz"]
    call = {"dgemm": oz.gemm, "zgemm": oz.zgemm, "noalloc": oz.gemm_noalloc}[c["kind"]]
    call(c["ta"], c["tb"], c["m"], c["n"], c["k"], c["alpha"], state["A"], state["lda"], state["B"], state["ldb"], c["beta"],
         state["C"], state["ldc"], c["s"])
    return state["C"]


def work(case):
    """Operands read once, C written once (and read where beta is not 0); the int8 operations of the s products
    that the caller asked for (3 s for complex data), for a batch those of the 16 moduli that most entries need."""
    if case["kind"] == "batch":
        rng = np.random.default_rng([case["count"], case["lo"], case["hi"]])
        nbytes = ops = 0
        for _ in range(case["count"]):
            m, n, k = (int(round(math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]))))) for _ in range(3))
            if case["ops"] == "mixed":
                rng.integers(2), rng.integers(2)
            nbytes += 8 * (m * k + k * n + m * n)
            ops += 2 * m * n * k * 16
        return {"bytes": nbytes, "flops": ops}
    m, n, k = case["m"], case["n"], case["k"]
    elem, planes = (16, 3 * case["s"]) if case["kind"] == "zgemm" else (8, case["s"])
    return {"bytes": elem * (m * k + k * n + m * n * (2 if case["beta"] else 1)), "flops": 2.0 * m * n * k * planes}


def _op(X, ld, rows, op, cplx):
    """the matrix op(X) of a flat column-major buffer whose stored matrix has `rows` rows"""
    X = torch.view_as_complex(X.view(-1, 2)) if cplx else X
    M = X.view(-1, ld)[:, :rows].T
    M = M if op == "N" else M.T
    return (M.conj().resolve_conj() if op == "C" else M).contiguous()


def exact(case, seed):
    if case["kind"] == "batch":
        probs, C = _batch_problems(case, seed)
        for p in probs:
            a = _op(p["A"], p["lda"], p["lda"], p["ta"], False)
            b = _op(p["B"], p["ldb"], p["ldb"], p["tb"], False)
            p["C"].copy_((a @ b).T.reshape(-1))
        return C
    (A, lda), (B, ldb), (C, ldc) = _gemm_inputs(case, seed)
    m, n, k, cplx = case["m"], case["n"], case["k"], case["kind"] == "zgemm"
    a = _op(A, lda, m if case["ta"] == "N" else k, case["ta"], cplx)
    b = _op(B, ldb, k if case["tb"] == "N" else n, case["tb"], cplx)
    full = torch.view_as_complex(C.view(-1, 2)) if cplx else C
    view = full.view(n, ldc)[:, :m]
    view.copy_(case["alpha"] * (a @ b).T + (case["beta"] * view if case["beta"] else 0))
    return C
