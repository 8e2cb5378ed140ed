"""Timed cases of the dense-solve library: what a user's program has it do,
through the device entry points of the `lmx` package (torch tensors in HBM).

Families, each over the sizes and options it is used with:
  matmul  C = alpha op(A) op(B) + beta C in FP64, FP32, BF16 and FP32 on
          split-BF16 tiles, any transposes, ragged shapes
  gram    A^T A and A A^T (matMulAtAP, the normal equations)
  lu      luSolve: factor and solve in FP64, the factors and pivots kept
  chol    choleskySolve: the same for a symmetric positive definite matrix
  mixed   FP32 factor with refinement to FP64 accuracy, LU and Cholesky
  factor  a new right-hand side for a factor that stays in HBM
  batch   thousands of independent solves of uneven order in one launch

An entry point that overwrites its inputs (the factorisations do) gets them
restored from the caller's copy at the start of a pass, on the device.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "linear-massiv_amd"))

import lmx  # noqa: E402


def listed():
    return [
        # a small product inside a larger program: one launch's latency
        {"name": "matmul_100", "family": "matmul", "dtype": "f64", "ta": "N", "tb": "N", "m": 100, "n": 100, "k": 100,
         "beta": 0.0},
        # accumulating into a result with a transposed operand, odd sizes
        {"name": "matmul_odd", "family": "matmul", "dtype": "f64", "ta": "T", "tb": "N", "m": 1999, "n": 1001,
         "k": 777, "beta": 1.0},
        # a large double-precision product
        {"name": "matmul_8192", "family": "matmul", "dtype": "f64", "ta": "N", "tb": "N", "m": 8192, "n": 8192,
         "k": 8192, "beta": 0.0},
        # a large product on the BF16 matrix cores
        {"name": "matmul_bf16", "family": "matmul", "dtype": "bf16", "ta": "N", "tb": "N", "m": 8192, "n": 8192,
         "k": 8192, "beta": 0.0},
        # luSolve of a small system, one right-hand side: latency
        {"name": "lu_100", "family": "lu", "n": 100, "nrhs": 1},
        # luSolve at the order the CPU library is used at
        {"name": "lu_500", "family": "lu", "n": 500, "nrhs": 1},
        # luSolve and choleskySolve of a large system, several right-hand sides
        {"name": "lu_8192", "family": "lu", "n": 8192, "nrhs": 16},
        {"name": "chol_8192", "family": "chol", "n": 8192, "nrhs": 16},
        # the largest solves: FP32 factor, FP64 refinement
        {"name": "lu_mixed_16384", "family": "mixed", "kind": "lu", "n": 16384, "nrhs": 1},
        {"name": "chol_mixed_4096", "family": "mixed", "kind": "chol", "n": 4096, "nrhs": 64},
        # a new right-hand side for a resident factor
        {"name": "factor_4096", "family": "factor", "kind": "lu", "n": 4096, "nrhs": 1},
        # many independent systems of uneven order, half LU, half Cholesky
        {"name": "batch_8000", "family": "batch", "count": 4000, "n_max": 512, "precision": "f64"},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    family = rng.choice(["matmul", "matmul", "gram", "lu", "lu", "chol", "chol", "mixed", "factor", "batch"])
    if family == "matmul":
        return {"family": family, "dtype": rng.choice(["f64", "f64", "f32", "bf16", "bf16x3"]),
                "ta": rng.choice("NNT"), "tb": rng.choice("NNT"), "m": _log(rng, 16, 8192), "n": _log(rng, 16, 8192),
                "k": _log(rng, 16, 8192), "beta": rng.choice([0.0, 0.0, 1.0, -0.5])}
    if family == "gram":
        return {"family": family, "trans": rng.choice("TTN"), "n": _log(rng, 16, 6000), "k": _log(rng, 16, 8192)}
    if family in ("lu", "chol"):
        return {"family": family, "n": _log(rng, 16, 8192), "nrhs": _log(rng, 1, 32)}
    if family == "mixed":
        return {"family": family, "kind": rng.choice(["lu", "chol"]), "n": _log(rng, 256, 12000),
                "nrhs": rng.choice([1, 1, 2, 7, 16, 64])}
    if family == "factor":
        return {"family": family, "kind": rng.choice(["lu", "chol"]), "n": _log(rng, 64, 8192),
                "nrhs": _log(rng, 1, 32)}
    return {"family": family, "count": _log(rng, 100, 4000), "n_max": _log(rng, 32, 512),
            "precision": rng.choice(["f64", "f32"])}


# ---------------------------------------------------------------- inputs

def _uniform(shape, g, dtype=torch.float64):
    return torch.rand(shape, dtype=dtype, device="cuda", generator=g) * 2 - 1


def _signs(shape, g):
    return torch.randint(0, 2, shape, device="cuda", generator=g).to(torch.float64) * 2 - 1


def _cosines(n):
    """The orthogonal n x n DCT-II matrix."""
    i = torch.arange(n, dtype=torch.int64, device="cuda")
    out = torch.empty((n, n), dtype=torch.float64, device="cuda")
    for r in range(0, n, 4096):  # in slices: the angles of n = 16384 are 2 GiB each way
        angle = (i[r:r + 4096, None] * (2 * i[None, :] + 1)) % (4 * n)
        out[r:r + 4096] = torch.cos(angle.to(torch.float64) * (math.pi / (2 * n)))
    out *= math.sqrt(2.0 / n)
    out[0] *= math.sqrt(0.5)
    return out


def _general(count, n, g):
    """count dense n x n systems that need row interchanges in every column:
    iid U[-1, 1] entries plus a dense orthogonal matrix with random row and
    column signs, large enough that the condition number stays below 10."""
    A = _uniform((count, n, n), g)
    left, right = _signs((count, n, 1), g), _signs((count, 1, n), g)
    Q = _cosines(n) * (1.5 * math.sqrt(n))
    for c in range(count):
        A[c].addcmul_(Q * left[c], right[c])
    return A


def _spd(count, n, g):
    """count matrices G G^T / n + I, G iid N(0, 1)."""
    G = torch.randn((count, n, n), dtype=torch.float64, device="cuda", generator=g)
    A = torch.bmm(G, G.transpose(1, 2).contiguous()) / n
    A.diagonal(dim1=1, dim2=2).add_(1.0)
    return A


def _system(kind, n, g):
    return (_general if kind == "lu" else _spd)(1, n, g)[0]


def _batch_shapes(case):
    """LU problems then Cholesky problems, order log-uniform in [8, n_max],
    1 to 8 right-hand sides; problems of one order lie next to each other.
    The shapes are the case's (a plan is made for them), the values the seed's."""
    r = np.random.default_rng(case["count"])
    shapes = []
    for kind in (lmx.BATCH_LU, lmx.BATCH_CHOLESKY):
        n = np.exp(r.uniform(np.log(8), np.log(case["n_max"]), case["count"])).round().astype(int)
        shapes += sorted(zip([kind] * case["count"], n.tolist(), r.integers(1, 9, case["count"]).tolist()))
    return shapes


def _groups(probs):
    """(first, last + 1) of each run of problems of one kind and order."""
    i = 0
    while i < len(probs):
        j = i
        while j < len(probs) and (probs[j].kind, probs[j].n) == (probs[i].kind, probs[i].n):
            j += 1
        yield i, j
        i = j


def _data(case, seed):
    """The inputs alone (torch tensors in HBM), from the seed."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    f = case["family"]
    if f == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        dt = torch.float64 if case["dtype"] == "f64" else torch.float32
        d = {"A": _uniform((k, m) if case["ta"] == "T" else (m, k), g, dt),
             "B": _uniform((n, k) if case["tb"] == "T" else (k, n), g, dt), "C0": _uniform((m, n), g, dt)}
        if case["dtype"] == "bf16":
            d["A"], d["B"] = d["A"].bfloat16(), d["B"].bfloat16()
        return d
    if f == "gram":
        n, k = case["n"], case["k"]
        return {"A": _uniform((k, n) if case["trans"] == "T" else (n, k), g)}
    if f == "batch":
        probs, na, nb, npiv = lmx.batch_layout(_batch_shapes(case))
        A = torch.empty(na, dtype=torch.float64, device="cuda")
        for i, j in _groups(probs):
            n, at = probs[i].n, probs[i].a_offset
            block = (_general if probs[i].kind == lmx.BATCH_LU else _spd)(j - i, n, g)
            A[at:at + block.numel()] = block.reshape(-1)
        return {"probs": probs, "A": A, "B": _uniform((nb,), g), "npiv": npiv}
    kind = case.get("kind", f)
    return {"A": _system(kind, case["n"], g), "B": _uniform((case["n"], case["nrhs"]), g)}


def prepare(case, seed):
    d = _data(case, seed)
    d["case"] = case
    f = case["family"]
    i32 = {"dtype": torch.int32, "device": "cuda"}
    if f == "matmul":
        d["C"] = torch.empty_like(d["C0"])
    elif f == "gram":
        d["C"] = torch.empty((case["n"], case["n"]), dtype=torch.float64, device="cuda")
    elif f in ("lu", "chol"):
        d["LU"], d["X"] = torch.empty_like(d["A"]), torch.empty_like(d["B"])
        d["ipiv"], d["info"] = torch.zeros(case["n"], **i32), torch.zeros(1, **i32)
    elif f == "mixed":
        d["X"] = torch.empty_like(d["B"])
    elif f == "factor":
        d["X"] = torch.empty_like(d["B"])
        d["factor"] = lmx.Factor(d["A"], lmx.FACTOR_LU if case["kind"] == "lu" else lmx.FACTOR_CHOLESKY)
    elif f == "batch":
        count = len(d["probs"])
        d["plan"] = lmx.BatchPlan(d["probs"], d["A"].numel(), d["B"].numel(), d["npiv"],
                                  lmx.PREC_F64 if case["precision"] == "f64" else lmx.PREC_F32, lmx.BATCH_GRAPH)
        d["work"] = torch.empty_like(d["A"]) if case["precision"] == "f64" else d["A"]
        d["X"] = torch.empty_like(d["B"])
        d["ipiv"], d["info"] = torch.zeros(d["npiv"], **i32), torch.zeros(count, **i32)
        d["iterations"] = torch.zeros(count, **i32)
    return d


_GEMM = {"f64": lmx.dgemm_dev, "f32": lmx.sgemm_dev, "bf16": lmx.gemm_bf16_dev, "bf16x3": lmx.sgemm_bf16x3_dev}


def run(state):
    case = state["case"]
    f = case["family"]
    if f == "matmul":
        if case["beta"] != 0.0:
            state["C"].copy_(state["C0"])
        _GEMM[case["dtype"]](state["A"], state["B"], state["C"], beta=case["beta"], transa=case["ta"],
                             transb=case["tb"])
        return state["C"]
    if f == "gram":
        lmx.syrk_dev(state["A"], state["C"], trans=case["trans"])
        return state["C"]
    if f in ("lu", "chol"):
        state["LU"].copy_(state["A"])
        state["X"].copy_(state["B"])
        if f == "lu":
            lmx.gesv_dev(state["LU"], state["ipiv"], state["X"], state["info"])
            return {"x": state["X"], "factors": state["LU"], "ipiv": state["ipiv"], "info": state["info"]}
        lmx.posv_dev(state["LU"], state["X"], state["info"])
        return {"x": state["X"], "factors": state["LU"], "info": state["info"]}
    if f == "mixed":
        solve = lmx.gesv_mixed_dev if case["kind"] == "lu" else lmx.posv_mixed_dev
        r = solve(state["A"], state["B"], state["X"])
        return {"x": state["X"], "info": int(r.info), "converged": int(r.converged)}
    if f == "factor":
        state["factor"].solve_dev(state["B"], state["X"])
        return state["X"]
    if state["work"] is not state["A"]:  # the FP64 path factors in place
        state["work"].copy_(state["A"])
    state["X"].copy_(state["B"])
    state["plan"].execute(state["work"], state["X"], state["info"], state["ipiv"], state["iterations"])
    return {"x": state["X"], "info": state["info"]}


def work(case):
    f = case["family"]
    if f == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        size = {"f64": 8, "f32": 4, "bf16x3": 4, "bf16": 2}[case["dtype"]]
        out = 8 if case["dtype"] == "f64" else 4
        return {"bytes": (m * k + k * n) * size + m * n * out * (2 if case["beta"] else 1), "flops": 2.0 * m * n * k}
    if f == "gram":
        n, k = case["n"], case["k"]
        return {"bytes": 8 * (n * k + n * n), "flops": float(n) * (n + 1) * k}
    if f == "batch":
        # E[n^2] and E[n^3] of n log-uniform in [8, n_max], 4.5 right-hand sides on average
        top, span = case["n_max"], math.log(case["n_max"] / 8.0)
        n2, n3 = (top ** 2 - 64) / (2 * span), (top ** 3 - 512) / (3 * span)
        pairs = case["count"]
        written = 2 if case["precision"] == "f64" else 1  # the FP64 path leaves its factors
        return {"bytes": 8 * pairs * n2 * (written + 0.5 * written), "flops": pairs * (n3 + 2 * 2 * n2 * 4.5)}
    n, r = case["n"], case["nrhs"]
    if f == "factor":
        return {"bytes": 8 * (n * n * (1.0 if case["kind"] == "lu" else 0.5) + 2 * n * r), "flops": 2.0 * n * n * r}
    lu = case.get("kind", f) == "lu"
    read = n * n * (1.0 if lu else 0.5)
    return {"bytes": 8 * (read * (1 if f == "mixed" else 2) + 2 * n * r),
            "flops": (2.0 if lu else 1.0) * n ** 3 / 3 + 2.0 * n * n * r}


def exact(case, seed):
    d = _data(case, seed)
    f = case["family"]
    if f == "matmul":
        A = d["A"].double().t().contiguous() if case["ta"] == "T" else d["A"].double()
        B = d["B"].double().t().contiguous() if case["tb"] == "T" else d["B"].double()
        return A @ B + case["beta"] * d["C0"].double()
    if f == "gram":
        At = d["A"].t().contiguous()
        return At @ d["A"] if case["trans"] == "T" else d["A"] @ At
    if f == "batch":
        X = torch.empty_like(d["B"])
        for i, j in _groups(d["probs"]):
            ps = d["probs"][i:j]
            n, at = ps[0].n, ps[0].a_offset
            A = d["A"][at:at + (j - i) * n * n].view(j - i, n, n)
            B = torch.zeros((j - i, n, 8), dtype=torch.float64, device="cuda")
            for c, p in enumerate(ps):
                B[c, :, :p.nrhs] = d["B"][p.b_offset:p.b_offset + n * p.nrhs].view(n, p.nrhs)
            S = torch.linalg.solve(A, B)
            for c, p in enumerate(ps):
                X[p.b_offset:p.b_offset + n * p.nrhs] = S[c, :, :p.nrhs].reshape(-1)
        return {"x": X, "info": None}
    X = torch.linalg.solve(d["A"], d["B"])
    if f == "factor":
        return X
    if f == "mixed":
        return {"x": X, "info": None, "converged": None}
    return {"x": X, "factors": None, "info": None, "ipiv": None} if f == "lu" else {"x": X, "factors": None,
                                                                                    "info": None}
