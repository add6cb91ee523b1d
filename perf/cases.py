"""The calls that programs built on this library make, with their sizes.

A tensor of k column-major m x n matrices is the contiguous torch tensor of
shape (k, n, m), as everywhere in ``gputils_amd.api``.  Every case names an
``op``:

  projection   one projected-gradient step y = P (x - a g) with the norm and
               the inner product that its stopping test reads (axpy,
               nullspace_project, nrm2, dot)
  posv         fused FP64 Cholesky factorisation and solve
  chol         Cholesky factorisation, then the solve from the factor
  mixed        FP32 Cholesky with FP64 refinement
  gemm         C = alpha A B + beta C in FP32, split BF16 and FP64
  gels         least squares of many equal tall systems
  qr           QR factorisation, least squares from the factors (Q^T b, then
               the triangular solve) and the explicit thin Q
  ragged       least squares of systems of uneven size through a plan
  svd          singular values with both sets of vectors
  nullspace    null-space basis and projector, and one projection with them

Calls that overwrite their input get it copied in first, as a program that
keeps its matrices has to.
"""
import math

import numpy as np
import torch

from gputils_amd import api

_DT = {"fp32": torch.float32, "bf16x3": torch.float32, "fp64": torch.float64}


def listed():
    return [
        # a controller's inner loop on a handful of problems: launches and host time
        {"name": "projection_16x96", "op": "projection", "k": 16, "m": 48, "n": 96, "r": 40, "dtype": "fp32"},
        # many small SPD systems (the 32 x 32 configuration)
        {"name": "posv_1024x32", "op": "posv", "k": 1024, "n": 32, "nrhs": 1, "dtype": "fp64"},
        # mid-size SPD systems through the factorise-then-solve interface
        {"name": "chol_256x200", "op": "chol", "k": 256, "n": 200, "nrhs": 1, "dtype": "fp64"},
        # the headline: 8192 SPD systems of 128, four right-hand sides
        {"name": "mixed_8192x128", "op": "mixed", "k": 8192, "n": 128, "nrhs": 4},
        # batched products of the 64^3 configuration, into a kept result
        {"name": "gemm_16384x64", "op": "gemm", "k": 16384, "m": 64, "n": 64, "kk": 64, "dtype": "fp32",
         "beta": 0.0, "out": True},
        # batched products of odd sizes in the split-BF16 mode, result allocated by the call
        {"name": "gemm_2000x100x75x50", "op": "gemm", "k": 2000, "m": 100, "n": 75, "kk": 50, "dtype": "bf16x3",
         "beta": 0.0, "out": False},
        # one large product in FP64, accumulated into a kept result
        {"name": "gemm_1500x1100x1300", "op": "gemm", "k": 1, "m": 1500, "n": 1100, "kk": 1300, "dtype": "fp64",
         "beta": 1.0, "out": True},
        # regression on many equal tall systems
        {"name": "gels_1024x100x30", "op": "gels", "k": 1024, "m": 100, "n": 30, "nrhs": 1, "dtype": "fp32"},
        # one tall matrix: factors, a solve and the basis (what the QR class does for a single matrix)
        {"name": "qr_1x600x150", "op": "qr", "k": 1, "m": 600, "n": 150, "nrhs": 1, "dtype": "fp64"},
        # 4096 systems of uneven size, one refinement step (the ragged configuration)
        {"name": "ragged_4096", "op": "ragged", "count": 4096, "nmin": 8, "nmax": 64, "mmax": 512, "steps": 1},
        # singular value decompositions with U and V
        {"name": "svd_512x80x50", "op": "svd", "k": 512, "m": 80, "n": 50, "dtype": "fp64"},
        # null spaces of 2048 rank-deficient 48 x 96 matrices (the SVD configuration)
        {"name": "nullspace_2048x48x96", "op": "nullspace", "k": 2048, "m": 48, "n": 96, "r": 40, "dtype": "fp32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _count(rng, one, budget, most):
    """A batch size between 1 and what the budget allows, by its logarithm."""
    return _log(rng, 1, max(1, min(most, int(budget / one))))


def draw(rng):
    op = rng.choice(["projection", "posv", "chol", "mixed", "gemm", "gemm", "gels", "qr", "ragged", "svd",
                     "nullspace"])
    dtype = rng.choice(["fp32", "fp64"])
    if op == "projection":
        n = _log(rng, 8, 160)
        m = rng.randint(max(1, n // 4), max(1, (3 * n) // 4))
        return {"op": op, "k": _count(rng, n * n, 2e7, 4096), "m": m, "n": n, "r": m, "dtype": dtype}
    if op == "posv":
        n = _log(rng, 4, 160)
        return {"op": op, "k": _count(rng, n ** 3, 3e9, 32768), "n": n, "nrhs": rng.randint(1, 6), "dtype": "fp64"}
    if op == "chol":
        n = _log(rng, 8, 400)
        return {"op": op, "k": _count(rng, n ** 3, 1.5e9, 16384), "n": n, "nrhs": rng.randint(1, 6), "dtype": dtype}
    if op == "mixed":
        n = _log(rng, 8, 128)
        return {"op": op, "k": _count(rng, n ** 3, 1.5e10, 16384), "n": n, "nrhs": rng.randint(1, 8)}
    if op == "gemm":
        mode = rng.choice(["fp32", "bf16x3", "fp64"])
        keep = rng.random() < 0.5
        beta = rng.choice([0.0, 1.0]) if keep else 0.0
        if rng.random() < 0.6:  # batches of small products
            m, n, kk = (_log(rng, 4, 160) for _ in range(3))
            k = _count(rng, 2.0 * m * n * kk + 60.0 * (m * n + m * kk + kk * n), 4e9, 16384)
        else:  # few large ones
            m, n, kk = (_log(rng, 128, 2000) for _ in range(3))
            k = _count(rng, 2.0 * m * n * kk, 6e9, 16)
        return {"op": op, "k": k, "m": m, "n": n, "kk": kk, "dtype": mode, "beta": beta, "out": keep}
    if op == "gels":
        n = _log(rng, 4, 100)
        m = n + max(8, n // 2) + rng.randint(0, 2 * n)
        return {"op": op, "k": _count(rng, m * n * n, 1e9, 8192), "m": m, "n": n, "nrhs": rng.randint(1, 4),
                "dtype": dtype}
    if op == "qr":
        n = _log(rng, 8, 200)
        m = n + max(8, n // 2) + rng.randint(0, 3 * n)
        return {"op": op, "k": _count(rng, m * n * n, 1.5e8, 64), "m": m, "n": n, "nrhs": rng.randint(1, 3),
                "dtype": dtype}
    if op == "ragged":
        nmax = rng.randint(16, 64)
        return {"op": op, "count": _log(rng, 16, 4096), "nmin": rng.randint(2, 12), "nmax": nmax,
                "mmax": rng.randint(2 * nmax, 512), "steps": rng.randint(1, 2)}
    if op == "svd":
        n = _log(rng, 4, 72)
        m = n + rng.randint(max(1, n // 4), n)
        return {"op": op, "k": _count(rng, float(m) * n * n * n, 3e9, 2048), "m": m, "n": n, "dtype": dtype}
    n = _log(rng, 8, 120)
    m = rng.randint(max(1, n // 4), max(1, (2 * n) // 3))
    r = m if dtype == "fp64" or m < 8 or rng.random() < 0.5 else m - rng.randint(1, m // 6)
    return {"op": op, "k": _count(rng, float(n) * m ** 3, 1.5e10, 2048), "m": m, "n": n, "r": r, "dtype": dtype}


# ---------------------------------------------------------------- inputs --
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)


def _reflect_rows(g, X, times=4):
    """Q X for every matrix of X (k, p, q), Q a product of random reflectors."""
    k, p, _ = X.shape
    for _ in range(times):
        v = _normal(g, k, p, 1)
        v /= v.norm(dim=1, keepdim=True)
        X = X - (2.0 * v) * (v * X).sum(dim=1, keepdim=True)
    return X


def _spd(g, k, n, decades, dtype):
    """SPD matrices Q diag(lambda) Q^T, lambda from 1 to 10^decades by its logarithm."""
    lam = torch.logspace(0, decades if n > 1 else 0, n, dtype=torch.float64, device="cuda")
    A = torch.empty(k, n, n, dtype=dtype, device="cuda")
    step = max(1, (1 << 25) // (n * n))
    for s in range(0, k, step):
        c = min(step, k - s)
        half = _reflect_rows(g, torch.diag(lam.sqrt()).expand(c, n, n))
        A[s:s + c] = (half @ half.transpose(1, 2).contiguous()).to(dtype)
    return A


def _low_rank(g, k, m, n, r, dtype):
    """m x n matrices of rank r, singular values U[0.1, 10], in (k, n, m) storage."""
    sig = 0.1 + 9.9 * torch.rand(k, r, generator=g, device="cuda", dtype=torch.float64)
    X = torch.zeros(k, n, m, dtype=torch.float64, device="cuda")
    X[:, torch.arange(r), torch.arange(r)] = sig
    X = _reflect_rows(g, X)
    return _reflect_rows(g, X.transpose(1, 2).contiguous()).transpose(1, 2).contiguous().to(dtype)


def _ragged_sizes(c):
    """Sizes and offsets of the systems: they belong to the case, as a program's plan does."""
    rng = np.random.default_rng([c["count"], c["nmin"], c["nmax"], c["mmax"]])
    ns = rng.integers(c["nmin"], c["nmax"] + 1, c["count"])
    lo = np.maximum(16, ns + 4)
    ms = np.minimum(lo + np.floor(rng.random(c["count"]) * (c["mmax"] - lo + 1)).astype(np.int64), c["mmax"])
    ms = np.maximum(ms, ns)
    oa = np.concatenate([[0], np.cumsum(ms * ns)[:-1]]).astype(np.int64)
    ob = np.concatenate([[0], np.cumsum(ms)[:-1]]).astype(np.int64)
    return ms.astype(np.int32), ns.astype(np.int32), oa, ob


def _inputs(c, seed):
    g, op = _gen(seed), c["op"]
    if op in ("projection", "nullspace"):
        dt = _DT[c["dtype"]]
        s = {"A": _low_rank(g, c["k"], c["m"], c["n"], c["r"], dt), "x": _normal(g, c["k"], 1, c["n"]).to(dt)}
        if op == "projection":
            s["g"] = _normal(g, c["k"], 1, c["n"]).to(dt)
        return s
    if op in ("posv", "chol", "mixed"):
        dt = _DT[c.get("dtype", "fp64")]
        A = _spd(g, c["k"], c["n"], 4.0 if op == "mixed" else 2.0, dt)
        return {"A": A, "B": _normal(g, c["k"], c["nrhs"], c["n"]).to(dt)}
    if op == "gemm":
        dt = _DT[c["dtype"]]

        def unit(*shape):
            return (2.0 * torch.rand(*shape, generator=g, device="cuda", dtype=dt) - 1.0).contiguous()
        s = {"A": unit(c["k"], c["kk"], c["m"]), "B": unit(c["k"], c["n"], c["kk"])}
        if c["out"]:
            s["C"] = unit(c["k"], c["n"], c["m"])
        return s
    if op in ("gels", "qr"):
        dt = _DT[c["dtype"]]
        return {"A": _normal(g, c["k"], c["n"], c["m"]).to(dt), "B": _normal(g, c["k"], c["nrhs"], c["m"]).to(dt)}
    if op == "svd":
        return {"A": _normal(g, c["k"], c["n"], c["m"]).to(_DT[c["dtype"]])}
    ms, ns, oa, ob = _ragged_sizes(c)
    total = int((ms.astype(np.int64) * ns).sum())
    return {"ms": ms, "ns": ns, "oa": oa, "ob": ob, "A": _normal(g, total), "B": _normal(g, int(ms.sum()))}


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    op = case["op"]
    if op == "projection":
        s["N"], _, s["rank"] = api.nullspace_batched(s["A"])
        s["y"] = torch.empty_like(s["x"])
    elif op in ("posv", "chol", "gels", "qr"):
        s["a"], s["b"] = torch.empty_like(s["A"]), torch.empty_like(s["B"])
        s["info"] = torch.empty(case["k"], dtype=torch.int32, device="cuda")
        if op == "qr":
            k, m, n = case["k"], case["m"], case["n"]
            s["eye"] = torch.eye(m, dtype=s["A"].dtype, device="cuda")[:n].expand(k, n, m).contiguous()
            s["q"] = torch.empty_like(s["eye"])
    elif op == "mixed":
        s["X"] = torch.empty_like(s["B"])
    elif op == "gemm" and case["out"]:
        s["c"] = torch.empty_like(s["C"])
    elif op == "nullspace":
        s["y"] = torch.empty_like(s["x"])
    elif op == "ragged":
        s["plan"] = api.RaggedLeastSquares(s["ms"], s["ns"], s["oa"], s["ob"])
        s["b"] = torch.empty_like(s["B"])
    return s


# ------------------------------------------------------------------ runs --
def run(s):
    c = s["case"]
    op = c["op"]
    if op == "projection":
        y = s["y"]
        y.copy_(s["x"])
        api.axpy(-0.125, s["g"], y)
        api.nullspace_project(s["N"], s["rank"], y)
        return {"y": y, "norm": api.nrm2(y), "slope": api.dot(y, s["g"])}
    if op == "posv":
        s["a"].copy_(s["A"])
        s["b"].copy_(s["B"])
        api.posv_batched(s["a"], s["b"], s["info"])
        return {"L": s["a"], "X": s["b"], "info": s["info"]}
    if op == "chol":
        s["a"].copy_(s["A"])
        s["b"].copy_(s["B"])
        info = api.potrf_batched(s["a"], s["info"])
        api.potrs_batched(s["a"], s["b"])
        return {"L": s["a"], "X": s["b"], "info": info}
    if op == "mixed":
        # the refinement steps each system took are a matter of rounding, not a result
        X, _, info = api.posv_mixed_batched(s["A"], s["B"], s["X"], tol=1e-12, max_iter=30)
        return {"X": X, "info": info}
    if op == "gemm":
        mode = "bf16x3" if c["dtype"] == "bf16x3" else "fp32"
        if not c["out"]:
            return {"C": api.gemm_batched(s["A"], s["B"], mode=mode)}
        if c["beta"] != 0.0:
            s["c"].copy_(s["C"])
        return {"C": api.gemm_batched(s["A"], s["B"], s["c"], beta=c["beta"], mode=mode)}
    if op == "gels":
        s["a"].copy_(s["A"])
        s["b"].copy_(s["B"])
        info = api.gels_batched(s["a"], s["b"], s["info"])
        return {"QR": s["a"], "X": s["b"], "info": info}
    if op == "qr":
        s["a"].copy_(s["A"])
        s["b"].copy_(s["B"])
        s["q"].copy_(s["eye"])
        tau = api.geqrf_batched(s["a"])
        api.ormqr_batched(s["a"], tau, s["b"], trans=True)
        api.trsm_upper_batched(s["a"], s["b"])
        api.ormqr_batched(s["a"], tau, s["q"], trans=False)
        return {"QR": s["a"], "tau": tau, "X": s["b"], "Q": s["q"]}
    if op == "ragged":
        s["b"].copy_(s["B"])
        return {"X": s["plan"](s["A"], s["b"], refine_steps=c["steps"])}
    if op == "svd":
        S, U, VT, info = api.gesvd_batched(s["A"], compute_u=True)
        return {"S": S, "U": U, "VT": VT, "info": info}
    N, P, rank = api.nullspace_batched(s["A"])
    s["y"].copy_(s["x"])
    out = {"P": P, "rank": rank, "y": api.nullspace_project(N, rank, s["y"])}
    if c["r"] == c["m"]:
        # with a deficient rank the columns of N are any basis of the null space: y and P pin the space
        out["N"] = N
    return out


# ------------------------------------------------------------------ work --
def work(case):
    c, op = case, case["op"]
    if op == "ragged":
        ms, ns, _, _ = _ragged_sizes(c)
        ms, ns = ms.astype(np.float64), ns.astype(np.float64)
        flops = 2 * ms * ns ** 2 - 2 * ns ** 3 / 3 + (1 + c["steps"]) * 6 * ms * ns
        return {"bytes": float(8 * (ms * ns + ms + ns).sum()), "flops": float(flops.sum())}
    k, n, m = float(c["k"]), float(c["n"]), float(c.get("m", c["n"]))
    es = 8.0 if c.get("dtype", "fp64") == "fp64" else 4.0
    nr = float(c.get("nrhs", 1))
    tri = n * (n + 1) / 2
    if op == "projection":
        q = n - c["r"]
        return {"bytes": es * k * (n * q + 3 * n), "flops": k * (4 * n * q + 6 * n)}
    if op in ("posv", "chol"):
        return {"bytes": es * k * (2 * tri + 2 * n * nr), "flops": k * (n ** 3 / 3 + 2 * n * n * nr)}
    if op == "mixed":
        return {"bytes": 8 * k * (tri + 2 * n * nr), "flops": k * (n ** 3 / 3 + 6 * n * n * nr)}
    if op == "gemm":
        kk = float(c["kk"])
        return {"bytes": es * k * (m * kk + kk * n + (1 + (c["beta"] != 0.0)) * m * n), "flops": 2 * k * m * n * kk}
    fact = 2 * m * n * n - 2 * n ** 3 / 3
    if op == "gels":
        return {"bytes": es * k * (2 * m * n + (m + n) * nr), "flops": k * (fact + (4 * m * n - n * n) * nr)}
    if op == "qr":
        return {"bytes": es * k * (3 * m * n + n + (m + n) * nr), "flops": k * (2 * fact + (4 * m * n - n * n) * nr)}
    if op == "svd":
        # QR, eight Jacobi sweeps on R with V, U from the reflectors
        return {"bytes": es * k * (m * n + n + m * m + n * n),
                "flops": k * (fact + 8 * 9 * n ** 3 + 4 * m * m * n - 2 * m * n * n)}
    q = n - c["r"]
    fact = 2 * n * m * m - 2 * m ** 3 / 3
    return {"bytes": es * k * (m * n + 2 * n * n + 2 * n),
            "flops": k * (fact + 8 * 9 * m ** 3 + 4 * n * n * m - 2 * n * m * m + n * n * q + 4 * n * q)}


# ----------------------------------------------------------------- exact --
def _mats(t):
    """(k, n, m) storage on the GPU -> (k, m, n) matrices in 64 bits on the host."""
    return t.cpu().double().transpose(1, 2).contiguous().numpy()


def _store(x):
    return np.ascontiguousarray(np.swapaxes(x, 1, 2))


def exact(case, seed):
    c, op = case, case["op"]
    s = _inputs(c, seed)
    if op in ("projection", "nullspace"):
        A = _mats(s["A"])
        U, sig, VT = np.linalg.svd(A, full_matrices=True)
        n, r = c["n"], c["r"]
        V2 = np.swapaxes(VT, 1, 2)[:, :, r:]
        V2T = np.ascontiguousarray(np.swapaxes(V2, 1, 2))
        x = _mats(s["x"])
        if op == "projection":
            g = _mats(s["g"])
            y = V2 @ (V2T @ (x - 0.125 * g))
            return {"y": _store(y), "norm": np.array([math.sqrt((y * y).sum())]),
                    "slope": np.array([(y * g).sum()])}
        out = {"P": _store(V2 @ V2T), "rank": None, "y": _store(V2 @ (V2T @ x))}
        if r == c["m"]:
            Q, R = np.linalg.qr(np.swapaxes(A, 1, 2), mode="complete")
            N = np.zeros((c["k"], n, n))
            N[:, :, :n - r] = Q[:, :, r:]
            out["N"] = _store(N)
        return out
    if op in ("posv", "chol", "mixed"):
        A, B = _mats(s["A"]), _mats(s["B"])
        A = np.tril(A) + np.swapaxes(np.tril(A, -1), 1, 2)
        X = _store(np.linalg.solve(A, B))
        if op == "mixed":
            return {"X": X, "info": None}
        L = np.linalg.cholesky(A) + np.triu(_mats(s["A"]), 1)  # the upper triangle stays as it was
        return {"L": _store(L), "X": X, "info": None}
    if op == "gemm":
        A, B = _mats(s["A"]), _mats(s["B"])
        C = A @ B
        if c["beta"] != 0.0:
            C += c["beta"] * _mats(s["C"])
        return {"C": _store(C)}
    if op in ("gels", "qr"):
        A, B = _mats(s["A"]), _mats(s["B"])
        h, tau = np.linalg.qr(A, mode="raw")  # LAPACK's packed factors, (k, n, m) as stored
        Q, R = np.linalg.qr(A)
        QT = np.ascontiguousarray(np.swapaxes(Q, 1, 2))
        if op == "gels":
            X = B.copy()
            X[:, :c["n"]] = np.linalg.solve(R, QT @ B)
            return {"QR": h, "X": _store(X), "info": None}
        # below the solution the right-hand side holds the rest of Q^T b
        Qc, _ = np.linalg.qr(A, mode="complete")
        X = np.swapaxes(Qc, 1, 2) @ B
        X[:, :c["n"]] = np.linalg.solve(R, QT @ B)
        return {"QR": h, "tau": tau, "X": _store(X), "Q": _store(Q)}
    if op == "svd":
        A = _mats(s["A"])
        k, m, n = A.shape
        _, sig, VT = np.linalg.svd(A, full_matrices=False)
        V = np.swapaxes(VT, 1, 2)
        top = np.take_along_axis(V, np.abs(V).argmax(axis=1)[:, None, :], axis=1)
        V = V * -np.sign(top)  # the largest entry of each v is negative
        Q, _ = np.linalg.qr(A, mode="complete")
        U = np.concatenate([(A @ V) / sig[:, None, :], Q[:, :, n:]], axis=2)
        return {"S": sig[:, None, :], "U": _store(U), "VT": V, "info": None}
    A, B = s["A"].cpu().numpy(), s["B"].cpu().numpy()
    X = B.copy()
    for m, n, oa, ob in zip(s["ms"], s["ns"], s["oa"], s["ob"]):
        a = A[oa:oa + int(m) * int(n)].reshape(int(n), int(m)).T
        q, r = np.linalg.qr(a)
        X[ob:ob + n] = np.linalg.solve(r, q.T @ B[ob:ob + m])
    return {"X": X}
