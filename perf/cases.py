"""Workloads of the HPD factor-and-solve library, as its users' programs run
them: single solves from one diagonal block to n = 16384, resident factors,
mixed precision with refinement, uneven batches, inverses and single triangular
solves.

listed() holds the fixed cases, draw() one more of the same ranges, prepare()
builds a case's inputs and plans on the GPU, run() is one pass through the
public entry points, work() the bytes and operations a pass cannot do
without, exact() the same outputs from torch in 64 bits.

Matrices are Gram matrices of normal data with a ridge, G G^T / n + shift I:
the covariance and kernel matrices such solvers are given.  shift sets the
condition number (about (4 + shift) / shift).
"""
from __future__ import annotations

import math

import numpy as np
import torch

import elemental_amd as E
from elemental_amd.batch import BatchPlan, uneven_sizes
from elemental_amd.mixed import IROptions, workspace_bytes


def listed():
    return [
        # one small system, as a filter or a fitting step solves it thousands
        # of times in a row: latency and launches
        {"name": "solve_n96", "do": "solve", "n": 96, "k": 1, "uplo": "L", "dtype": "f64", "pad": 0, "shift": 1.0},
        # a medium system with a few right-hand sides (the smallest size of the benchmark family)
        {"name": "solve_n2048", "do": "solve", "n": 2048, "k": 16, "uplo": "L", "dtype": "f64", "pad": 0, "shift": 1.0},
        # an odd size in a padded buffer whose upper triangle is stored
        {"name": "solve_n3001_upper", "do": "solve", "n": 3001, "k": 5, "uplo": "U", "dtype": "f64", "pad": 6,
         "shift": 0.1},
        # single precision throughout
        {"name": "solve_n4000_f32", "do": "solve", "n": 4000, "k": 8, "uplo": "L", "dtype": "f32", "pad": 0,
         "shift": 1.0},
        # the largest: the benchmark's size in plain FP64
        {"name": "solve_n16384", "do": "solve", "n": 16384, "k": 32, "uplo": "L", "dtype": "f64", "pad": 0,
         "shift": 0.1},
        # a factor kept resident, solved with again for new right-hand sides
        {"name": "after_n8192", "do": "after", "n": 8192, "k": 8, "uplo": "L", "pad": 0, "shift": 0.1},
        # the mixed-precision solve with its default options, ragged
        {"name": "mixed_n5003", "do": "mixed", "n": 5003, "k": 3, "trailing": "f32", "refine": "ir", "shift": 0.01},
        # the mixed-precision solve as the benchmark runs it
        {"name": "mixed_n16384", "do": "mixed", "n": 16384, "k": 32, "trailing": "bf16x3", "refine": "cg",
         "shift": 0.001},
        # many small systems of uneven size in one launch sequence, FP64 and
        # FP32 with FP64 refinement
        {"name": "batch_f64", "do": "batch", "count": 1024, "lo": 16, "hi": 1024, "kmax": 8, "precision": "f64",
         "sizes": 4, "shift": 0.1},
        {"name": "batch_f32", "do": "batch", "count": 1024, "lo": 16, "hi": 1024, "kmax": 8, "precision": "f32",
         "sizes": 5, "shift": 0.1},
        # the inverse of a covariance matrix (a precision matrix)
        {"name": "inverse_n3000", "do": "inverse", "n": 3000, "uplo": "L", "pad": 0, "shift": 0.1},
        # sampling from a Gaussian with the factor at hand: one triangular
        # solve with a block of vectors
        {"name": "trsm_n4100", "do": "trsm", "n": 4100, "k": 64, "trans": "T", "pad": 1, "shift": 0.1},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    do = rng.choice(["solve", "solve", "solve", "after", "mixed", "mixed", "batch", "inverse", "trsm"])
    pad = rng.choice([0, 0, 1, 6, 32])
    uplo = rng.choice(["L", "L", "L", "U"])
    shift = rng.choice([1.0, 0.1, 0.01])
    if do == "solve":
        dtype = rng.choice(["f64", "f64", "f32"])
        return {"do": do, "n": _log_int(rng, 16, 16000), "k": _log_int(rng, 1, 32), "uplo": uplo, "dtype": dtype,
                "pad": pad, "shift": 1.0 if dtype == "f32" else shift}
    if do == "after":
        return {"do": do, "n": _log_int(rng, 64, 12000), "k": _log_int(rng, 1, 32), "uplo": uplo, "pad": pad,
                "shift": shift}
    if do == "mixed":
        return {"do": do, "n": _log_int(rng, 512, 16000), "k": _log_int(rng, 1, 32),
                "trailing": rng.choice(["f32", "bf16x3"]), "refine": rng.choice(["ir", "cg"]),
                "shift": rng.choice([0.1, 0.01, 0.001])}
    if do == "batch":
        return {"do": do, "count": _log_int(rng, 32, 1000), "lo": 16, "hi": _log_int(rng, 64, 1024),
                "kmax": rng.randint(1, 8), "precision": rng.choice(["f64", "f32"]), "sizes": rng.randint(10, 10**6),
                "shift": 0.1}
    if do == "inverse":
        return {"do": do, "n": _log_int(rng, 64, 4000), "uplo": uplo, "pad": pad, "shift": shift}
    return {"do": do, "n": _log_int(rng, 128, 8000), "k": _log_int(rng, 2, 64), "trans": rng.choice(["N", "T"]),
            "pad": pad, "shift": shift}


# ---------------------------------------------------------------- inputs
_DTYPE = {"f64": torch.float64, "f32": torch.float32}


def _gram(n, shift, gen):
    G = torch.randn(n, n, dtype=torch.float64, device="cuda", generator=gen)
    A = G @ G.t()
    del G
    A.div_(n)
    A.diagonal().add_(shift)
    return A  # symmetric


def _matrix(height, width, pad=0, dtype=torch.float64):
    return E.Matrix(height, width, height + pad, dtype=dtype)


def _filled(t, pad=0, dtype=torch.float64):
    M = _matrix(t.shape[0], t.shape[1], pad, dtype)
    M.tensor().copy_(t)
    return M


def _sizes(case):
    return uneven_sizes(case["count"], case["lo"], case["hi"], case["kmax"], case["sizes"])


def _inputs(case, seed):
    """The case's numbers: A (and B), or lists of them for a batch."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["do"] == "batch":
        As, Bs = [], []
        for n, k in zip(*_sizes(case)):
            As.append(_gram(int(n), case["shift"], gen))
            Bs.append(torch.randn(int(n), int(k), dtype=torch.float64, device="cuda", generator=gen))
        return As, Bs
    n = case["n"]
    A = _gram(n, case["shift"], gen)
    B = None if case["do"] == "inverse" else torch.randn(n, case["k"], dtype=torch.float64, device="cuda",
                                                         generator=gen)
    return A, B


def _uplo(case):
    return E.UPPER if case.get("uplo") == "U" else E.LOWER


def prepare(case, seed):
    A, B = _inputs(case, seed)
    do = case["do"]
    if do == "batch":
        plan = BatchPlan(*_sizes(case), precision=case["precision"])
        A0, B0 = plan.empty_a(), plan.empty_b()
        for i in range(len(A)):
            plan.a_view(A0, i).copy_(A[i])
            plan.b_view(B0, i).copy_(B[i])
        return {"case": case, "plan": plan, "A0": A0, "B0": B0, "A": A0.clone(), "B": B0.clone()}
    pad = case.get("pad", 0)
    dt = _DTYPE[case.get("dtype", "f64")]
    s = {"case": case, "uplo": _uplo(case)}
    if do in ("solve", "inverse"):  # these overwrite A: the program keeps its own and works on a copy
        s["A0"] = _filled(A, pad, dt)
        s["A"] = _matrix(case["n"], case["n"], pad, dt)
    else:
        s["A"] = _filled(A, pad, dt)
    del A
    if do in ("after", "trsm"):  # the resident factor
        E.Cholesky(s["uplo"], s["A"])
    if B is not None:
        s["B0"] = _filled(B, pad, dt)
        s["B"] = _matrix(case["n"], case["k"], pad, dt)
    if do == "mixed":
        s["opts"] = IROptions(trailing=case["trailing"], refine=case["refine"])
        s["work"] = torch.empty(workspace_bytes(case["n"], case["k"], s["opts"]), dtype=torch.uint8, device="cuda")
    return s


# ------------------------------------------------------------------ pass
def run(s):
    case = s["case"]
    do = case["do"]
    if do == "batch":
        s["B"].copy_(s["B0"])
        if case["precision"] == "f64":
            s["A"].copy_(s["A0"])
            s["plan"].solve(s["A"], s["B"])
            return s["A"], s["B"]
        s["plan"].solve(s["A"], s["B"])
        return s["B"]
    if do in ("solve", "inverse"):
        s["A"].tensor().copy_(s["A0"].tensor())
    if do == "inverse":
        E.HPDInverse(s["uplo"], s["A"])
        return s["A"].tensor()
    s["B"].tensor().copy_(s["B0"].tensor())
    if do == "solve":
        E.HPDSolve(s["uplo"], E.NORMAL, s["A"], s["B"])
        return s["A"].tensor(), s["B"].tensor()
    if do == "after":
        E.SolveAfter(s["uplo"], E.NORMAL, s["A"], s["B"])
    elif do == "mixed":
        rep = E.HPDSolveMixed(s["A"], s["B"], s["opts"], s["work"])
        if not rep.converged:
            raise RuntimeError("the mixed solve did not converge")
    else:
        E.Trsm(E.LEFT, E.LOWER, E.TRANSPOSE if case["trans"] == "T" else E.NORMAL, E.NON_UNIT, 1.0, s["A"], s["B"])
    return s["B"].tensor()


def work(case):
    do = case["do"]
    if do == "batch":
        n, k = (v.astype(np.float64) for v in _sizes(case))
        tri, nk = n * (n + 1) / 2, n * k
        # the plain solve writes the factor, the refined one reads A again for a residual
        return {"bytes": float((16 * tri + 16 * nk).sum()),
                "flops": float((n**3 / 3 + 2 * n * n * k).sum())}
    n = float(case["n"])
    tri = n * (n + 1) / 2
    size = 4 if case.get("dtype") == "f32" else 8
    if do == "inverse":
        return {"bytes": 2 * size * tri, "flops": n**3}
    k = float(case["k"])
    if do == "solve":
        return {"bytes": 2 * size * tri + 2 * size * n * k, "flops": n**3 / 3 + 2 * n * n * k}
    if do == "mixed":
        return {"bytes": size * tri + 2 * size * n * k, "flops": n**3 / 3 + 2 * n * n * k}
    solves = 2 if do == "after" else 1
    return {"bytes": size * tri + 2 * size * n * k, "flops": solves * n * n * k}


# ----------------------------------------------------------- 64-bit values
def _factor_in(A, upper):
    """The factor in its triangle of A, A's own values in the other one."""
    L = torch.linalg.cholesky(A)
    return torch.triu(L.t()) + torch.tril(A, -1) if upper else torch.tril(L) + torch.triu(A, 1)


def exact(case, seed):
    A, B = _inputs(case, seed)
    do = case["do"]
    if do == "batch":
        plan = BatchPlan(*_sizes(case), precision=case["precision"])
        Ax, Bx = plan.empty_a(), plan.empty_b()
        for i in range(len(A)):
            L = torch.linalg.cholesky(A[i])
            plan.a_view(Ax, i).copy_(torch.tril(L) + torch.triu(A[i], 1))
            plan.b_view(Bx, i).copy_(torch.cholesky_solve(B[i], L))
        return (Ax, Bx) if case["precision"] == "f64" else Bx
    upper = case.get("uplo") == "U"
    if case.get("dtype") == "f32":
        A, B = A.float().double(), B.float().double()
        A = torch.triu(A) + torch.triu(A, 1).t() if upper else torch.tril(A) + torch.tril(A, -1).t()
    if do == "inverse":
        X = torch.cholesky_inverse(torch.linalg.cholesky(A))
        return torch.triu(X) + torch.tril(A, -1) if upper else torch.tril(X) + torch.triu(A, 1)
    if do == "solve":
        return _factor_in(A, upper), torch.cholesky_solve(B, torch.linalg.cholesky(A))
    L = torch.linalg.cholesky(A)
    del A
    if do == "trsm":
        return torch.linalg.solve_triangular(L.t() if case["trans"] == "T" else L, B, upper=case["trans"] == "T")
    return torch.cholesky_solve(B, L)
