"""The work that programs have this library do, as cases that a timing program can run.

A case is a dict of plain values with an "op"; listed() holds the fixed ones, draw(rng) makes more of the
same ranges, prepare / run / work / exact take either.  Matrices and vectors are on the GPU, column-major,
as the C ABI takes them; a flat column-major rows x cols buffer is held as a torch tensor (cols, ld).

The inputs are the reference harness's phi-mode distribution, (r1 - 0.5) exp(phi sqrt(-2 ln r1) sin(2 pi r2))
with r1, r2 uniform: phi sets the range of the exponents, and with it the number of slices.
"""
import math
import random

import numpy as np
import torch

import ozblas_amd
from ozblas_amd.autograd import ozaki_matmul

DEVICE = "cuda:0"
GIB = 1 << 30


def listed():
    return [
        # a short inner product of a serving loop or a small solver: launches and latency
        {"name": "ddot_1003", "op": "dot", "prec": "d", "n": 1003, "phi": 1.0, "sum": 1},
        # the inner product of a large solver (the benchmark's DDOT)
        {"name": "ddot_1e6", "op": "dot", "prec": "d", "n": 1000000, "phi": 2.0, "sum": 1},
        # dense matrix-vector product of an iterative method (the benchmark's DGEMV)
        {"name": "dgemv_8192", "op": "gemv", "prec": "d", "trans": "N", "m": 8192, "n": 8192, "phi": 0.5, "sum": 1},
        # one sparse product with a matrix split once, as a solver of the user's own calls it
        {"name": "dcsrmv_laplace100", "op": "csrmv", "prec": "d", "matrix": "laplace", "grid": 100, "presplit": True,
         "phi": 1.0, "sum": 1},
        # a whole reproducible conjugate-gradient solve (the benchmark's, with fewer iterations)
        {"name": "dcg_laplace100", "op": "cg", "prec": "d", "grid": 100, "iters": 250, "sum": 1},
        # a small reproducible DGEMM in the plain form: bitwise the CPU library's result
        {"name": "dgemm_fp64_256", "op": "gemm", "prec": "d", "form": "fp64", "ta": "N", "tb": "N", "m": 256, "n": 256,
         "k": 256, "phi": 1.0, "sum": 1, "pad": 0},
        # the plain form at an ordinary size, uneven: FP64 matrix cores and the sum over the slice pairs
        {"name": "dgemm_fp64_2500", "op": "gemm", "prec": "d", "form": "fp64", "ta": "T", "tb": "N", "m": 2500,
         "n": 2301, "k": 2700, "phi": 1.0, "sum": 1, "pad": 0},
        # the headline product: correctly rounded DGEMM on INT8 matrix cores
        {"name": "dgemm_int8_8192", "op": "gemm", "prec": "d", "form": "int8", "ta": "N", "tb": "N", "m": 8192,
         "n": 8192, "k": 8192, "phi": 0.5, "sum": 1, "pad": 0},
        # the same form on ragged, padded, transposed operands of a wide exponent range
        {"name": "dgemm_int8_ragged", "op": "gemm", "prec": "d", "form": "int8", "ta": "N", "tb": "T", "m": 2001,
         "n": 1777, "k": 3001, "phi": 4.0, "sum": 1, "pad": 3},
        # binary32 with the library's default ordered sum
        {"name": "sgemm_1100", "op": "gemm", "prec": "s", "form": "fp64", "ta": "N", "tb": "N", "m": 1000, "n": 1100,
         "k": 1200, "phi": 1.0, "sum": 0, "pad": 0},
        # many uneven products in one call, the plan kept by the handle from call to call
        {"name": "batched_256", "op": "batched", "form": "int8", "count": 256, "lo": 64, "hi": 1024, "sizes": 4,
         "phi": 2.0},
        # a training step's product and its two gradients: forward INT8, backward FP16 (the defaults)
        {"name": "autograd_2048", "op": "autograd", "m": 2048, "k": 1024, "n": 2048, "phi": 1.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: op, type and options by use, sizes over the logarithm of their range."""
    op = rng.choice(["dot", "dot", "gemv", "csrmv", "cg", "gemm", "gemm", "gemm", "gemm", "batched", "autograd"])
    phi = rng.choice([0.5, 1.0, 2.0, 4.0])
    if op == "dot":
        return {"op": rng.choice(["dot", "dot", "nrm2"]), "prec": rng.choice(["d", "d", "d", "s"]),
                "n": _log(rng, 100, 4000000), "phi": phi, "sum": rng.choice([1, 1, 0])}
    if op == "gemv":
        prec = rng.choice(["d", "d", "d", "s", "ds"])
        return {"op": op, "prec": prec, "trans": rng.choice("NT"), "m": _log(rng, 65, 9500), "n": _log(rng, 65, 9500),
                "phi": min(phi, 2.0), "sum": 0 if prec == "ds" else rng.choice([1, 1, 0])}
    if op == "csrmv":
        matrix = rng.choice(["laplace", "rows"])
        return {"op": op, "prec": rng.choice(["d", "d", "s"]), "matrix": matrix, "grid": _log(rng, 10, 110),
                "presplit": rng.choice([True, True, False]), "phi": min(phi, 2.0), "sum": rng.choice([1, 0])}
    if op == "cg":
        return {"op": op, "prec": rng.choice(["d", "d", "s"]), "grid": _log(rng, 12, 100), "iters": _log(rng, 30, 200),
                "sum": rng.choice([1, 1, 0])}
    if op == "batched":
        lo = _log(rng, 24, 200)
        return {"op": op, "form": "int8", "count": _log(rng, 8, 256), "lo": lo, "hi": _log(rng, lo + 100, 1024),
                "sizes": rng.randrange(1000), "phi": phi}
    if op == "autograd":
        return {"op": op, "m": _log(rng, 150, 2500), "k": _log(rng, 150, 2500), "n": _log(rng, 150, 2500),
                "phi": min(phi, 2.0)}
    prec, form = rng.choice([("d", "int8"), ("d", "int8"), ("d", "int8"), ("d", "fp16"), ("d", "bf16"), ("d", "fp64"),
                             ("d", "fp64"), ("s", "fp64"), ("ds", "fp64")])
    top = 6500 if form == "int8" else 2600
    return {"op": "gemm", "prec": prec, "form": form, "ta": rng.choice("NT"), "tb": rng.choice("NT"),
            "m": _log(rng, 100, top), "n": _log(rng, 100, top), "k": _log(rng, 100, top), "phi": phi,
            "sum": 1 if form != "fp64" else 0 if prec != "d" else rng.choice([1, 1, 0]), "pad": rng.choice([0, 0, 1, 8])}


# ---- inputs ---------------------------------------------------------------------------------------
def _dtype(prec):
    return torch.float32 if prec == "s" else torch.float64


def _phi(gen, shape, phi, dtype=torch.float64):
    r1 = 1.0 - torch.rand(shape, generator=gen, device=DEVICE, dtype=torch.float64)
    r2 = torch.rand(shape, generator=gen, device=DEVICE, dtype=torch.float64)
    r2 = torch.sin(2.0 * math.pi * r2)
    return ((r1 - 0.5) * torch.exp(phi * torch.sqrt(-2.0 * torch.log(r1)) * r2)).to(dtype)


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _laplace(grid, dtype):
    """3-D 7-point Laplacian on a grid^3 grid, diagonal 6 + 1e-3, CSR with int32 indices, sorted columns."""
    n = grid ** 3
    idx = torch.arange(n, device=DEVICE, dtype=torch.int64)
    at = (idx % grid, (idx // grid) % grid, idx // (grid * grid))
    cols, vals, keep = [], [], []
    for axis, step in ((2, -1), (1, -1), (0, -1), (0, 0), (0, 1), (1, 1), (2, 1)):
        to = at[axis] + step
        keep.append((to >= 0) & (to < grid))
        cols.append(idx + step * grid ** axis)
        vals.append(torch.full((n,), -1.0 if step else 6.0 + 1e-3, device=DEVICE, dtype=torch.float64))
    keep, cols, vals = torch.stack(keep, 1), torch.stack(cols, 1), torch.stack(vals, 1)
    rowptr = torch.zeros(n + 1, device=DEVICE, dtype=torch.int64)
    rowptr[1:] = torch.cumsum(keep.sum(1), 0)
    return rowptr.to(torch.int32), cols[keep].to(torch.int32), vals[keep].to(dtype)


def _rows(gen, grid, phi, dtype):
    """A general sparse matrix of grid^3 rows: 0 to 24 entries a row, within a band of 2 grid^2 columns."""
    n = grid ** 3
    length = torch.randint(0, 25, (n,), generator=gen, device=DEVICE)
    rowptr = torch.zeros(n + 1, device=DEVICE, dtype=torch.int64)
    rowptr[1:] = torch.cumsum(length, 0)
    row = torch.repeat_interleave(torch.arange(n, device=DEVICE), length)
    off = torch.randint(-grid * grid, grid * grid + 1, (row.numel(),), generator=gen, device=DEVICE)
    return rowptr.to(torch.int32), (row + off).clamp(0, n - 1).to(torch.int32), _phi(gen, (row.numel(),), phi, dtype)


def _batch_sizes(case):
    rng = random.Random(case["sizes"])
    return [tuple(rng.randint(case["lo"], case["hi"]) for _ in range(3)) for _ in range(case["count"])]


def _gemm_inputs(case, gen):
    m, n, k, pad = case["m"], case["n"], case["k"], case["pad"]
    dtype = _dtype(case["prec"])
    ra, ca = (m, k) if case["ta"] == "N" else (k, m)
    rb, cb = (k, n) if case["tb"] == "N" else (n, k)
    A = _phi(gen, (ca, ra + pad), case["phi"], dtype)
    B = _phi(gen, (cb, rb + pad), case["phi"], dtype)
    return A, B


def _csr_inputs(case, gen):
    dtype = _dtype(case["prec"])
    if case["matrix"] == "laplace":
        rowptr, colind, val = _laplace(case["grid"], dtype)
    else:
        rowptr, colind, val = _rows(gen, case["grid"], case["phi"], dtype)
    return rowptr, colind, val, _phi(gen, (case["grid"] ** 3,), case["phi"], dtype)


def _cg_inputs(case, gen):
    dtype = _dtype(case["prec"])
    n = case["grid"] ** 3
    b = (2.0 * torch.rand((n,), generator=gen, device=DEVICE, dtype=torch.float64) - 1.0).to(dtype)
    return _laplace(case["grid"], dtype), b


def prepare(case, seed):
    gen = _generator(seed)
    op = case["op"]
    s = {"case": case}
    if op in ("dot", "nrm2"):
        s["x"], s["y"] = (_phi(gen, (case["n"],), case["phi"], _dtype(case["prec"])) for _ in range(2))
        s["handle"] = ozblas_amd.Handle(4 * GIB, sumMode=case["sum"])
    elif op == "gemv":
        m, n = case["m"], case["n"]
        dtype = _dtype(case["prec"])
        s["A"] = _phi(gen, (n, m), case["phi"], dtype)
        s["x"] = _phi(gen, (n if case["trans"] == "N" else m,), case["phi"], dtype)
        s["y"] = torch.zeros(m if case["trans"] == "N" else n, device=DEVICE, dtype=dtype)
        s["handle"] = ozblas_amd.Handle(16 * GIB, sumMode=case["sum"])
    elif op == "csrmv":
        s["rowptr"], s["colind"], s["val"], s["x"] = _csr_inputs(case, gen)
        s["y"] = torch.zeros_like(s["x"])
        s["handle"] = ozblas_amd.Handle(8 * GIB, sumMode=case["sum"])
        n = s["x"].numel()
        s["A"] = s["val"]
        if case["presplit"]:
            s["A"] = getattr(s["handle"], case["prec"] + "csrmv_splitA")(n, n, s["val"].numel(), s["val"], s["rowptr"])
    elif op == "cg":
        (s["rowptr"], s["colind"], s["val"]), s["b"] = _cg_inputs(case, gen)
        s["x"] = torch.zeros_like(s["b"])
        s["handle"] = ozblas_amd.Handle(4 * GIB, sumMode=case["sum"])
    elif op == "gemm":
        s["A"], s["B"] = _gemm_inputs(case, gen)
        s["C"] = torch.zeros((case["n"], case["m"]), device=DEVICE, dtype=_dtype(case["prec"]))
        s["handle"] = ozblas_amd.Handle(24 * GIB, sumMode=case["sum"], sliceType=case["form"])
    elif op == "batched":
        s["sizes"] = _batch_sizes(case)
        s["A"] = [_phi(gen, (k, m), case["phi"]) for m, n, k in s["sizes"]]
        s["B"] = [_phi(gen, (n, k), case["phi"]) for m, n, k in s["sizes"]]
        s["out"] = torch.zeros(sum(m * n for m, n, k in s["sizes"]), device=DEVICE, dtype=torch.float64)
        s["C"] = list(torch.split(s["out"], [m * n for m, n, k in s["sizes"]]))
        s["handle"] = ozblas_amd.Handle(GIB, sumMode=1, sliceType=case["form"])
    else:
        m, k, n = case["m"], case["k"], case["n"]
        s["A"] = _phi(gen, (m, k), case["phi"]).requires_grad_()
        s["B"] = _phi(gen, (k, n), case["phi"]).requires_grad_()
        s["W"] = torch.randn((m, n), generator=gen, device=DEVICE, dtype=torch.float64)
    torch.cuda.synchronize()
    return s


# ---- one pass -------------------------------------------------------------------------------------
def run(s):
    case = s["case"]
    op = case["op"]
    h = s.get("handle")
    if op == "dot":
        return getattr(h, case["prec"] + "dot")(case["n"], s["x"], s["y"])
    if op == "nrm2":
        return getattr(h, case["prec"] + "nrm2")(case["n"], s["x"])
    if op == "gemv":
        m, n = case["m"], case["n"]
        getattr(h, case["prec"] + "gemv")(case["trans"], m, n, 1.0, s["A"], m, s["x"], 0.0, s["y"])
        return s["y"]
    if op == "csrmv":
        n = s["x"].numel()
        getattr(h, case["prec"] + "csrmv")(n, n, s["val"].numel(), 1.0, s["A"], s["colind"], s["rowptr"], s["x"], 0.0,
                                           s["y"])
        return s["y"]
    if op == "cg":
        s["x"].zero_()
        history = getattr(h, case["prec"] + "cg")(s["b"].numel(), s["val"].numel(), s["val"], s["colind"], s["rowptr"],
                                                  s["b"], s["x"], case["iters"], 0.0)
        return {"x": s["x"], "history": history}
    if op == "gemm":
        getattr(h, case["prec"] + "gemm")(case["ta"], case["tb"], case["m"], case["n"], case["k"], 1.0, s["A"],
                                          s["A"].shape[1], s["B"], s["B"].shape[1], 0.0, s["C"], case["m"])
        return s["C"]
    if op == "batched":
        ms, ns, ks = ([x[i] for x in s["sizes"]] for i in range(3))
        one = len(ms)
        h.dgemm_batched(["N"] * one, ["N"] * one, ms, ns, ks, [1.0] * one, s["A"], ms, s["B"], ks, [0.0] * one, s["C"], ms)
        return s["out"]
    C = ozaki_matmul(s["A"], s["B"])
    dA, dB = torch.autograd.grad((C * s["W"]).sum(), (s["A"], s["B"]))
    return {"C": C.detach(), "dA": dA, "dB": dB}


# ---- what a pass cannot do without ------------------------------------------------------------------
def work(case):
    """Inputs read once, outputs written once; the multiply-adds of the product itself, whatever the slices add."""
    op = case["op"]
    size = 4 if case.get("prec") == "s" else 8
    if op in ("dot", "nrm2"):
        return {"bytes": size * case["n"] * (2 if op == "dot" else 1), "flops": 2 * case["n"]}
    if op == "gemv":
        m, n = case["m"], case["n"]
        return {"bytes": size * (m * n + m + n), "flops": 2 * m * n}
    if op in ("csrmv", "cg"):
        n = case["grid"] ** 3
        nnz = 7 * n - 6 * case["grid"] ** 2 if case.get("matrix") != "rows" else 12 * n
        product = (size + 4) * nnz + size * 2 * n + 4 * n
        if op == "csrmv":
            return {"bytes": product, "flops": 2 * nnz}
        # an iteration: the product, two dots, two updates that read two vectors and write one, and p
        return {"bytes": case["iters"] * (product + size * 10 * n), "flops": case["iters"] * (2 * nnz + 10 * n)}
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": size * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if op == "batched":
        return {"bytes": sum(8 * (m * k + k * n + m * n) for m, n, k in _batch_sizes(case)),
                "flops": sum(2 * m * n * k for m, n, k in _batch_sizes(case))}
    m, n, k = case["m"], case["n"], case["k"]
    return {"bytes": 8 * (3 * (m * k + k * n) + 4 * m * n), "flops": 6 * m * n * k}


# ---- the same in plain 64-bit torch and numpy -------------------------------------------------------
def _csr_product(rowptr, colind, val, x):
    rowptr, colind, val, x = (t.cpu().numpy() for t in (rowptr, colind, val.double(), x.double()))
    row = np.repeat(np.arange(len(x)), np.diff(rowptr))
    return np.bincount(row, weights=val * x[colind], minlength=len(x))


def exact(case, seed):
    gen = _generator(seed)
    op = case["op"]
    if op in ("dot", "nrm2"):
        x, y = (_phi(gen, (case["n"],), case["phi"], _dtype(case["prec"])).double() for _ in range(2))
        return float(x @ y) if op == "dot" else float(torch.sqrt(x @ x))
    if op == "gemv":
        A = _phi(gen, (case["n"], case["m"]), case["phi"], _dtype(case["prec"])).double()
        x = _phi(gen, (case["n"] if case["trans"] == "N" else case["m"],), case["phi"], _dtype(case["prec"])).double()
        return A.t() @ x if case["trans"] == "N" else A @ x
    if op == "csrmv":
        return _csr_product(*_csr_inputs(case, gen))
    if op == "cg":
        # the iterates follow the rounding of every step: only a whole solve in exact sums has this value
        return None
    if op == "gemm":
        A, B = (t.double() for t in _gemm_inputs(case, gen))
        m, n, k = case["m"], case["n"], case["k"]
        At = A[:, :m] if case["ta"] == "N" else A[:, :k].t()   # op(A) transposed, k x m
        Bt = B[:, :k] if case["tb"] == "N" else B[:, :n].t()   # op(B) transposed, n x k
        return Bt @ At
    if op == "batched":
        sizes = _batch_sizes(case)
        A = [_phi(gen, (k, m), case["phi"]) for m, n, k in sizes]
        B = [_phi(gen, (n, k), case["phi"]) for m, n, k in sizes]
        return torch.cat([(b @ a).reshape(-1) for a, b in zip(A, B)])
    A = _phi(gen, (case["m"], case["k"]), case["phi"])
    B = _phi(gen, (case["k"], case["n"]), case["phi"])
    W = torch.randn((case["m"], case["n"]), generator=gen, device=DEVICE, dtype=torch.float64)
    return {"C": A @ B, "dA": W @ B.t(), "dB": A.t() @ W}
