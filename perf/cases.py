"""The calls this framework is used for, as cases that can be timed and compared.

Whole solves from the smallest served order to the headline one (FP32, split
16-bit, both bandwidths, with and without eigenvectors), same-size and
mixed-size batches, and the stages that a program calls one by one: band
reduction on FP64 buffers, bulge chasing, the tridiagonal solver, and the back
transformation of a part of the eigenvectors.

A program keeps one context for many matrices, so one context per precision
is opened on first use and shared by all states.
"""
import math

import numpy as np
import torch

import evd4sc2025_amd as E

DEV = "cuda:0"
_PRECISION = {"fp32": E.PREC_FP32, "fp16": E.PREC_FP16, "bf16": E.PREC_BF16}
_contexts = {}


def _context(precision):
    if precision not in _contexts:
        ctx = E.Context(0)
        ctx.set_precision(_PRECISION[precision])
        _contexts[precision] = ctx
    return _contexts[precision]


def listed():
    return [
        # the order most requests of the serving mix have: launches and dependent steps count
        {"name": "eigh_256", "kind": "eigh", "n": 256, "b": 32, "nb": 256, "jobz": "V", "precision": "fp32"},
        # an ordinary matrix of no round size (a covariance, a graph Laplacian)
        {"name": "eigh_1000", "kind": "eigh", "n": 1000, "b": 32, "nb": 256, "jobz": "V", "precision": "fp32"},
        # a spectrum alone, of an odd order
        {"name": "values_3001", "kind": "eigh", "n": 3001, "b": 32, "nb": 256, "jobz": "N", "precision": "fp32"},
        # the mixed-precision form at an ordinary large order, ragged
        {"name": "eigh_fp16_5003", "kind": "eigh", "n": 5003, "b": 32, "nb": 1024, "jobz": "V", "precision": "fp16"},
        # the wide band of the precision form (b = 64), in its bfloat16 variant
        {"name": "eigh_bf16_b64_8192", "kind": "eigh", "n": 8192, "b": 64, "nb": 1024, "jobz": "V", "precision": "bf16"},
        # the headline solve
        {"name": "eigh_16384", "kind": "eigh", "n": 16384, "b": 32, "nb": 1024, "jobz": "V", "precision": "fp32"},
        # many small problems of one order (one layer's preconditioners, a batch of requests)
        {"name": "batch_32x256", "kind": "batch", "n": 256, "count": 32, "b": 32, "jobz": "V"},
        # small problems of many orders, every other one with eigenvectors
        {"name": "mixed_40", "kind": "mixed", "lo": 64, "hi": 2048, "count": 40},
        # stages as a program that owns its buffers calls them:
        # band -> tridiagonal
        {"name": "chase_6000", "kind": "chase", "n": 6000, "b": 32},
        # tridiagonal -> eigenvalues and vectors
        {"name": "tridiag_2500", "kind": "tridiag", "n": 2500},
        # full -> band on the double buffers of the reference's interface
        {"name": "band_f64_1500", "kind": "band_f64", "n": 1500, "b": 32, "nb": 256},
        # 1000 of 8192 eigenvectors from the tridiagonal's to the matrix's
        {"name": "vectors_8192x1000", "kind": "vectors", "n": 8192, "cols": 1000, "b": 32},
    ]


def _size(rng, lo, hi):
    """An order between lo and hi, even over its logarithm, half of them odd or ragged."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return n if rng.random() < 0.5 else max(lo, n // 64 * 64)


def draw(rng):
    kind = rng.choice(["eigh"] * 5 + ["batch", "mixed", "chase", "tridiag", "band_f64", "vectors"])
    if kind == "eigh":
        n = _size(rng, 64, 8192)
        return {"kind": kind, "n": n, "b": 64 if n >= 512 and rng.random() < 0.3 else 32, "nb": 256 if n < 4096 else 1024,
                "jobz": "N" if rng.random() < 0.3 else "V", "precision": rng.choice(["fp32", "fp32", "fp16", "bf16"])}
    if kind == "batch":
        n = _size(rng, 64, 1024)
        return {"kind": kind, "n": n, "count": rng.randint(2, max(4, min(48, 16384 // n))), "b": 32,
                "jobz": "N" if rng.random() < 0.3 else "V"}
    if kind == "mixed":
        return {"kind": kind, "lo": 64, "hi": _size(rng, 256, 2048), "count": rng.randint(8, 40)}
    if kind == "chase":
        return {"kind": kind, "n": _size(rng, 100, 10000), "b": rng.choice([32, 32, 64])}
    if kind == "tridiag":
        return {"kind": kind, "n": _size(rng, 100, 6000)}
    if kind == "band_f64":
        return {"kind": kind, "n": _size(rng, 200, 2500), "b": 32, "nb": 256}
    n = _size(rng, 1024, 8192) // 32 * 32
    return {"kind": kind, "n": n, "cols": rng.randint(1, n), "b": rng.choice([32, 32, 64])}


def _orders(case):
    """The orders of a mixed-size call: fixed by the case, log-uniform."""
    r = np.random.RandomState(case["count"] + case["hi"])
    return [int(round(x)) for x in np.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"]), case["count"]))]


def _symmetric(n, gen):
    """(X + X^T) / 2 with standard normal X, column-major on the GPU."""
    x = torch.randn(n, n, generator=gen, device=DEV)
    x += x.t().clone()
    x *= 0.5
    return x.t()


def _chase_reflectors(n, b, gen):
    """U as the bulge chase leaves it: sweep s, step j at rows s+1+jb.., ||u||^2 = 2."""
    steps = -(-(n - 1) // b)
    x = torch.randn(n, steps, b, generator=gen, device=DEV, dtype=torch.float64)
    s = torch.arange(n, device=DEV).view(n, 1, 1)
    k = torch.arange(steps * b, device=DEV).view(1, steps, b)
    x *= (k < n - 1 - s)
    length = (n - 1 - s - k[:, :, :1]).clamp(max=b)
    u = x / x.norm(dim=2, keepdim=True).clamp(min=1e-30)
    u[:, :, 0] += torch.where(u[:, :, 0] >= 0, 1.0, -1.0)
    u = u / u[:, :, :1].abs().sqrt()
    u = (u * (length >= 2)).view(n, steps * b)
    u[n - 2:] = 0.0
    at = torch.arange(n + b, device=DEV).view(1, -1) - torch.arange(n, device=DEV).view(-1, 1) - 1
    u = torch.where((at >= 0) & (at < steps * b), u.gather(1, at.clamp(0, steps * b - 1)), 0.0)
    return u.float().t()


def _panels(n, b, gen):
    """W, Y as the band reduction leaves them: panel p at row (p+1) b, column p b."""
    W, Y = E.colmajor(n, n, fill=0.0), E.colmajor(n, n, fill=0.0)
    for c in range(0, n - b - 1, b):
        m = n - b - c
        k = min(b, m)
        v = torch.randn(m, k, generator=gen, device=DEV, dtype=torch.float64).div_(math.sqrt(m)).tril_(-1)
        v.diagonal().fill_(1.0)
        g = v.t() @ v
        t = torch.linalg.inv(g.triu(1) + torch.diag(g.diagonal() / 2))
        W[c + b:, c:c + k] = (v @ t).float()
        Y[c + b:, c:c + k] = v.float()
    return W, Y


def prepare(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    kind = case["kind"]
    s = {"case": case, "ctx": _context(case.get("precision", "fp32"))}
    if kind == "eigh":
        s["A"] = _symmetric(case["n"], gen)
    elif kind == "batch":
        s["mats"] = [_symmetric(case["n"], gen) for _ in range(case["count"])]
    elif kind == "mixed":
        s["mats"] = [_symmetric(n, gen) for n in _orders(case)]
        s["jobz"] = ["V" if q % 2 else "N" for q in range(case["count"])]
    elif kind == "chase":
        n, b = case["n"], case["b"]
        band = torch.randn(n, 2 * b, generator=gen, device=DEV, dtype=torch.float64)
        off = torch.arange(2 * b, device=DEV).view(1, -1)
        band *= (off <= b) & (off + torch.arange(n, device=DEV).view(-1, 1) < n)
        s["band"], s["work"] = band.t(), torch.empty_like(band).t()
    elif kind == "tridiag":
        # the tridiagonal form of a Gaussian symmetric matrix
        n = case["n"]
        r = np.random.RandomState(seed % (1 << 32))
        s["D"] = torch.from_numpy(r.standard_normal(n)).to(DEV)
        s["E"] = torch.from_numpy(np.sqrt(r.chisquare(np.arange(n - 1, 0, -1)) / 2)).to(DEV)
    elif kind == "band_f64":
        n = case["n"]
        s["A"] = _symmetric(n, gen).double()
        s["work"] = E.colmajor(n, n, dtype=torch.float64)
        s["W"], s["Y"] = E.colmajor(n, n, dtype=torch.float64), E.colmajor(n, n, dtype=torch.float64)
    else:
        n, b = case["n"], case["b"]
        s["U"] = _chase_reflectors(n, b, gen)
        s["W"], s["Y"] = _panels(n, b, gen)
        s["Z"] = E.to_colmajor(torch.randn(n, case["cols"], generator=gen, device=DEV).div_(math.sqrt(n)))
        s["Zw"], s["Ww"] = E.colmajor(n, case["cols"]), E.colmajor(n, n)
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "eigh":
        r = E.syevd(ctx, s["A"], b=case["b"], nb=case["nb"], jobz=case["jobz"])
        return {"w": r.w, "Z": r.Z}
    if kind == "batch":
        w, Z = E.syevd_batched(ctx, s["mats"], b=case["b"], nb=256, jobz=case["jobz"])
        return {"w": w, "Z": Z}
    if kind == "mixed":
        return [{"w": r.w, "Z": r.Z} for r in E.syevd_mixed(ctx, s["mats"], jobz=s["jobz"], b=0)]
    if kind == "chase":
        # the chase consumes its band
        s["work"].copy_(s["band"])
        D, Eo, U = E.sb2st(ctx, s["work"], case["n"], case["b"])
        return {"D": D, "E": Eo, "U": U}
    if kind == "tridiag":
        w, Z = E.stedc(ctx, s["D"], s["E"])
        return {"w": w, "Z": Z}
    if kind == "band_f64":
        n, b = case["n"], case["b"]
        s["work"].copy_(s["A"])
        E.my_ZY_ZY_SBR_Vector(ctx, n, n, b, case["nb"], None, s["work"], s["W"], s["Y"])
        return {"B": s["work"].tril().triu(-b), "W": s["W"], "Y": s["Y"]}
    # the vectors replace their input and W's panels are merged in place
    s["Zw"].copy_(s["Z"])
    s["Ww"].copy_(s["W"])
    E.bc_back(ctx, s["Zw"], s["U"], case["n"], case["b"], 1)
    E.sbr_back(ctx, s["Zw"], s["Ww"], s["Y"], case["b"])
    return s["Zw"]


def _solve_work(n, jobz):
    # the two-stage solve's own count with eigenvectors, the reduction alone without
    return {"bytes": 4 * n * n * (2 if jobz == "V" else 1) + 8 * n, "flops": (10 if jobz == "V" else 4) / 3 * n ** 3}


def work(case):
    kind, n = case["kind"], case.get("n", 0)
    if kind == "eigh":
        return _solve_work(n, case["jobz"])
    if kind == "batch":
        return {k: v * case["count"] for k, v in _solve_work(n, case["jobz"]).items()}
    if kind == "mixed":
        each = [_solve_work(m, "V" if q % 2 else "N") for q, m in enumerate(_orders(case))]
        return {k: sum(e[k] for e in each) for k in ("bytes", "flops")}
    if kind == "chase":
        return {"bytes": 8 * n * (case["b"] + 1) + 4 * n * (n + case["b"]) + 16 * n, "flops": 6 * n * n * case["b"]}
    if kind == "tridiag":
        return {"bytes": 8 * n * n + 24 * n, "flops": 4 / 3 * n ** 3}
    if kind == "band_f64":
        return {"bytes": 8 * 4 * n * n, "flops": 4 / 3 * n ** 3}
    c = case["cols"]
    return {"bytes": 4 * (3 * n * n + 2 * n * c), "flops": 4 * n * n * c}


def _values(A):
    return torch.linalg.eigvalsh(A.double().cpu())


def exact(case, seed):
    kind, n = case["kind"], case.get("n", 0)
    if kind in ("eigh", "tridiag") and n > 3200 or kind == "chase":
        return None
    s = prepare(case, seed)
    # eigenvectors are defined up to their sign: only the values have an exact value
    if kind == "eigh":
        return {"w": _values(s["A"]), "Z": None}
    if kind == "batch":
        return {"w": torch.stack([_values(A) for A in s["mats"]]), "Z": None}
    if kind == "mixed":
        return [{"w": _values(A), "Z": None} for A in s["mats"]]
    if kind == "tridiag":
        T = torch.diag(s["D"]) + torch.diag(s["E"], -1)
        return {"w": _values(T), "Z": None}
    b = case["b"]
    if kind == "band_f64":
        A = s["A"].clone()
        W, Y = torch.zeros_like(A), torch.zeros_like(A)
        for c in range(0, n - b - 1, b):
            r = c + b
            k = min(b, n - r)
            P, tau = torch.geqrf(A[r:, c:c + b].clone())
            v = P[:, :k].tril(-1)
            v.diagonal().fill_(1.0)
            t = torch.zeros(k, k, dtype=A.dtype, device=A.device)
            g = v.t() @ v
            for j in range(k):
                t[:j, j] = -tau[j] * (t[:j, :j] @ g[:j, j])
                t[j, j] = tau[j]
            w = v @ t
            A[r:, c:c + b] = P.triu()
            A[c:c + b, r:] = P.triu().t()
            X = A[r:, r:] - (A[r:, r:] @ w) @ v.t()
            A[r:, r:] = X - v @ (w.t() @ X)
            W[r:, c:c + k], Y[r:, c:c + k] = w, v
        return {"B": A.tril().triu(-b), "W": W, "Y": Y}
    U = s["U"].double()
    Z = torch.zeros(n + b, case["cols"], dtype=torch.float64, device=DEV)
    Z[:n] = s["Z"]
    for sweep in range(n - 3, -1, -1):
        k = -(-(n - 1 - sweep) // b)
        u = U[sweep + 1:sweep + 1 + k * b, sweep].reshape(k, b, 1)
        rows = Z[sweep + 1:sweep + 1 + k * b].view(k, b, -1)
        rows -= u * (u * rows).sum(dim=1, keepdim=True)
    Z = Z[:n]
    W, Y = s["W"].double(), s["Y"].double()
    for c in reversed(range(0, n - b - 1, b)):
        Z[c + b:] -= W[c + b:, c:c + b] @ (Y[c + b:, c:c + b].t().contiguous() @ Z[c + b:])
    return Z
