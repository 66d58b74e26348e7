"""The work that programs give this library, as cases that can be timed.

Every case goes through the public entry points (the C API by its Python
binding) on inputs made from a seed.  Six paths stand for the uses:

gemm    a product whose operands are already in the HBM tile cache, as in a
        program that has used them before; the result is fetched to the host.
        FP64, FP32, complex, and FP64 accuracy from BF16 or FP8 products.
host    the drop-in replacement of a host BLAS: operands and result in
        ordinary host memory, nothing kept on the GPU between two calls.
normal  linear least squares by the normal equations: SYRK (HERK) and GEMM
        form them, POTRF factors, two TRSM solve.  Only the solution leaves
        the GPU.  All four of the library's main routines, chained.
posv    an SPD system solved by the reduced-precision factor with FP64
        iterative refinement.
sym     one step of a symmetric projection: SYMM, TRMM, SYR2K chained.
batch   an uneven batch of small products and triangular solves on device
        memory: a plan kept and replayed as a graph, or built on each call.
"""
import ctypes
import math
import random

import numpy as np
import torch

import xkblas_amd as xk

TORCH = {"s": torch.float32, "d": torch.float64, "c": torch.complex64, "z": torch.complex128}
NUMPY = {"s": np.float32, "d": np.float64, "c": np.complex64, "z": np.complex128}
REAL = {"s": torch.float32, "d": torch.float64, "c": torch.float32, "z": torch.float64}
SIZE = {"s": 4, "d": 8, "c": 8, "z": 16}
# what a program of each dense path already has in the tile cache
OPERANDS = {"gemm": ("A", "B", "C"), "normal": ("G", "Y"), "posv": ("A", "B"), "sym": ("A", "T", "B")}
OPS = {"N": xk.NoTrans, "T": xk.Trans, "C": xk.ConjTrans}


def listed():
    return [
        # a small ragged product: the cost of one call
        {"name": "gemm_d_small", "path": "gemm", "type": "d", "mode": 0, "op": "NN", "m": 230, "n": 187, "k": 301,
         "beta": 0.0},
        # FP64 on the matrix cores, no dimension a multiple of anything
        {"name": "gemm_d_ragged", "path": "gemm", "type": "d", "mode": 0, "op": "TN", "m": 5003, "n": 3001, "k": 9011,
         "beta": 0.0},
        # single precision
        {"name": "gemm_s", "path": "gemm", "type": "s", "mode": 0, "op": "NT", "m": 4096, "n": 4100, "k": 8192,
         "beta": 0.0},
        # FP64-accurate product from BF16 products at the benchmark's size
        {"name": "gemm_d_split_bf16", "path": "gemm", "type": "d", "mode": 2, "op": "NN", "m": 16384, "n": 16384,
         "k": 16384, "beta": -0.5},
        # the reference's own test case, called like a host BLAS
        {"name": "host_gemm_d", "path": "host", "type": "d", "m": 2048, "n": 2048, "k": 2048},
        # least squares: a small system, where launches count
        {"name": "normal_d_small", "path": "normal", "type": "d", "mode": 0, "uplo": "L", "trans": True, "n": 517,
         "k": 1500, "r": 9},
        # a large one
        {"name": "normal_d_large", "path": "normal", "type": "d", "mode": 0, "uplo": "L", "trans": False, "n": 8192,
         "k": 16384, "r": 64},
        # a complex one
        {"name": "normal_z", "path": "normal", "type": "z", "mode": 0, "uplo": "U", "trans": True, "n": 2048,
         "k": 4096, "r": 200},
        # SPD solve with refinement
        {"name": "posv_ir", "path": "posv", "uplo": "L", "n": 8192, "r": 64},
        # the symmetric and triangular products
        {"name": "sym_d", "path": "sym", "type": "d", "uplo": "L", "n": 4000, "r": 1900},
        # the uneven batch of the benchmark's ranges, as a replayed graph
        {"name": "batch_d", "path": "batch", "type": "d", "gemms": 4096, "trsms": 1024, "lo": 16, "hi": 512,
         "solve_lo": 32, "solve_hi": 1024, "r": 64, "shapes": 2027, "kept": True},
        # a small single-precision batch put together on each call
        {"name": "batch_s_small", "path": "batch", "type": "s", "gemms": 200, "trsms": 40, "lo": 16, "hi": 160,
         "solve_lo": 32, "solve_hi": 250, "r": 33, "shapes": 2028, "kept": False},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    path = rng.choice(["gemm", "gemm", "gemm", "host", "normal", "normal", "posv", "sym", "batch", "batch"])
    if path == "gemm":
        t, mode = rng.choice([("d", 0), ("d", 0), ("s", 0), ("z", 0), ("c", 0), ("d", 2), ("d", 2), ("d", 3)])
        lo, hi = (1000, 10000) if mode else {"d": (100, 8192), "s": (100, 10000), "z": (64, 4096), "c": (64, 5000)}[t]
        ops = "NT" if t in "sd" else "NTC"
        return {"path": path, "type": t, "mode": mode, "op": rng.choice(ops) + rng.choice(ops), "m": size(lo, hi),
                "n": size(lo, hi), "k": size(lo, hi), "beta": rng.choice([0.0, -0.5])}
    if path == "host":
        return {"path": path, "type": rng.choice("ds"), "m": size(200, 4000), "n": size(200, 4000),
                "k": size(200, 4000)}
    if path == "normal":
        t = rng.choice("ddsz")
        n = size(100, 2500 if t == "z" else 8000)
        return {"path": path, "type": t, "mode": rng.choice([0, 0, 2]) if t == "d" else 0, "uplo": rng.choice("LU"),
                "trans": rng.random() < 0.5, "n": n, "k": int(n * rng.uniform(2.0, 4.0)), "r": size(1, 500)}
    if path == "posv":
        return {"path": path, "uplo": rng.choice("LU"), "n": size(500, 8192), "r": size(1, 200)}
    if path == "sym":
        t = rng.choice("ddsz")
        return {"path": path, "type": t, "uplo": rng.choice("LU"), "n": size(100, 2500 if t == "z" else 5000),
                "r": size(50, 2000)}
    return {"path": path, "type": rng.choice("ds"), "gemms": size(20, 4096), "trsms": size(5, 1024),
            "lo": size(8, 32), "hi": size(100, 512), "solve_lo": size(16, 64), "solve_hi": size(200, 1024),
            "r": rng.choice([1, 17, 33, 64, 64, 100]), "shapes": rng.randrange(10000), "kept": rng.random() < 0.7}


# ---------------------------------------------------------------- inputs
def _matrix(g, m, n, t):
    """An m x n column-major matrix on the GPU, entries uniform in (-0.5, 0.5)."""
    x = torch.rand((n, m) + ((2,) if t in "cz" else ()), generator=g, device="cuda", dtype=REAL[t]) - 0.5
    return (torch.view_as_complex(x) if t in "cz" else x).T


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _inputs(case, seed):
    """The operands of a dense case, on the GPU."""
    g, path = _generator(seed), case["path"]
    if path in ("gemm", "host"):
        m, n, k, t = case["m"], case["n"], case["k"], case["type"]
        ta, tb = case.get("op", "NN")
        A = _matrix(g, *((m, k) if ta == "N" else (k, m)), t)
        B = _matrix(g, *((k, n) if tb == "N" else (n, k)), t)
        C = _matrix(g, m, n, t)
        if case.get("mode"):
            # rows of op(A) and columns of op(B) of widely different sizes
            sa = torch.exp2(torch.rand(m, generator=g, device="cuda", dtype=torch.float64) * 16 - 8)
            sb = torch.exp2(torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * 16 - 8)
            A *= sa[:, None] if ta == "N" else sa[None, :]
            B *= sb[None, :] if tb == "N" else sb[:, None]
        return {"A": A, "B": B, "C": C}
    if path == "normal":
        n, k, t = case["n"], case["k"], case["type"]
        return {"G": _matrix(g, *((k, n) if case["trans"] else (n, k)), t), "Y": _matrix(g, k, case["r"], t)}
    if path == "posv":
        n = case["n"]
        G = _matrix(g, n, n, "d")
        A = G @ G.T
        A.diagonal().add_(n)
        return {"A": A, "B": _matrix(g, n, case["r"], "d")}
    n, t = case["n"], case["type"]
    return {"A": _matrix(g, n, n, t), "T": _matrix(g, n, n, t), "B": _matrix(g, n, case["r"], t)}


class _Pinned:
    """Host memory of xkblas_malloc; what the tile cache holds of it goes with it."""

    def __init__(self, nbytes):
        self.nbytes = max(nbytes, 64)
        self.ptr = xk.lib().xkblas_malloc(self.nbytes)
        if not self.ptr:
            raise MemoryError("xkblas_malloc")
        self.__array_interface__ = {"data": (self.ptr, False), "shape": (self.nbytes,), "typestr": "|u1", "version": 3}

    def __del__(self):
        if getattr(self, "ptr", None):
            xk.lib().xkblas_memory_invalidate(self.ptr)
            xk.lib().xkblas_free(self.ptr, self.nbytes)


def _host(m, n, t):
    dt = np.dtype(NUMPY[t])
    return np.asarray(_Pinned(m * n * dt.itemsize))[:m * n * dt.itemsize].view(dt).reshape((m, n), order="F")


def _to_host(x, t):
    h = _host(*x.shape, t)
    torch.from_numpy(h.T).copy_(x.T)
    return h


def _keep_resident(t, *operands):
    """Brings matrices into the tile cache by a use of each (a product with one vector)."""
    for X in operands:
        v, y = np.zeros((X.shape[1], 1), NUMPY[t], order="F"), np.zeros((X.shape[0], 1), NUMPY[t], order="F")
        xk.gemm(xk.NoTrans, xk.NoTrans, 1.0, X, v, 0.0, y)
        for z in (v, y):
            xk.lib().xkblas_memory_invalidate(z.ctypes.data)


def _fetch(*results):
    for X, uplo in results:
        xk.lib().xkblas_memory_coherent_async(uplo, 0, X.shape[0], X.shape[1], X.ctypes.data, X.shape[0], X.itemsize)
    xk.lib().xkblas_sync()


class _Batch:
    """Problems on device memory: the flat pools of operands, and the list of problems."""

    def __init__(self, case, seed):
        t, self.r = case["type"], case["r"]
        self.gemms, self.solves = _shapes(case)
        g, dt, code = _generator(seed), TORCH[t], {"d": 0, "s": 1}[t]

        def pool(sizes):
            offs = np.concatenate([[0], np.cumsum([(x + 63) // 64 * 64 for x in sizes])]).astype(int)
            return offs, torch.rand(int(offs[-1]) + 64, generator=g, device="cuda", dtype=dt) - 0.5

        self.oa, self.A = pool([m * k for m, n, k in self.gemms])
        self.ob, self.B = pool([k * n for m, n, k in self.gemms])
        self.oc, self.C = pool([m * n for m, n, k in self.gemms])
        self.ol, self.L = pool([n * n for n in self.solves])
        self.ox, self.X = pool([n * self.r for n in self.solves])
        # unit-size diagonals, small entries below: a solve can be repeated
        # on its own result without growing or vanishing
        if self.solves:
            n = torch.tensor(self.solves, device="cuda")
            o = torch.tensor(self.ol, device="cuda")
            owner = torch.bucketize(torch.arange(len(self.L), device="cuda"), o[1:], right=True)
            self.L *= (0.5 / n.to(dt))[owner.clamp(max=len(self.solves) - 1)]
            del owner
            at = torch.cat([int(b) + torch.arange(s, device="cuda") * (s + 1) for b, s in zip(self.ol, self.solves)])
            self.L[at] = torch.where(self.L[at] < 0, -1.0, 1.0).to(dt)
        es = self.A.element_size()
        pa, pb, pc, pl, px = (x.data_ptr() for x in (self.A, self.B, self.C, self.L, self.X))
        probs = [xk.BatchProblem(xk.BATCH_GEMM, code, xk.NoTrans, xk.NoTrans, m, n, k, 1.5, -0.5,
                                 pa + int(self.oa[i]) * es, m, pb + int(self.ob[i]) * es, k,
                                 pc + int(self.oc[i]) * es, m) for i, (m, n, k) in enumerate(self.gemms)]
        probs += [xk.BatchProblem(xk.BATCH_TRSM, code, xk.NoTrans, xk.NoTrans, n, self.r, n, 1.0, 0.0,
                                  pl + int(self.ol[i]) * es, n, None, 0, px + int(self.ox[i]) * es, n)
                  for i, n in enumerate(self.solves)]
        self.count = len(probs)
        self.array = (xk.BatchProblem * self.count)(*probs)
        self.problems = ctypes.cast(self.array, ctypes.c_void_p)
        self.plan = None

    def __del__(self):
        if getattr(self, "plan", None):
            xk.lib().xkblas_batch_destroy(self.plan)


def _shapes(case):
    r = random.Random(case["shapes"])

    def size(lo, hi):
        return int(round(2 ** r.uniform(math.log2(lo), math.log2(hi))))

    gemms = [tuple(size(case["lo"], case["hi"]) for _ in range(3)) for _ in range(case["gemms"])]
    return gemms, [size(case["solve_lo"], case["solve_hi"]) for _ in range(case["trsms"])]


def prepare(case, seed):
    L = xk.lib()
    L.xkblas_init()
    L.xkblas_set_modemath(case.get("mode", 0))
    path, t = case["path"], case.get("type", "d")
    s = {"case": case}
    if path == "batch":
        s["batch"] = b = _Batch(case, seed)
        torch.cuda.synchronize()
        if case["kept"]:
            b.plan = L.xkblas_batch_create(b.problems, b.count)
            L.xkblas_batch_use_graph(b.plan, 1)
        return s
    x = _inputs(case, seed)
    if path == "host":
        for k, v in x.items():
            s[k] = np.asfortranarray(np.empty(v.shape[::-1], NUMPY[t]).T)
            torch.from_numpy(s[k].T).copy_(v.T)
        return s
    for k in list(x):
        s[k] = _to_host(x.pop(k), t)
    if path == "normal":
        n = case["n"]
        s["S"], s["X"] = _host(n, n, t), _host(n, case["r"], t)
        s["S"][:] = 0
        _keep_resident(t, s["S"])
    if path == "sym":
        n = case["n"]
        s["X"], s["S"] = _host(n, case["r"], t), _host(n, n, t)
        s["S"][:] = 0
        _keep_resident(t, s["S"])
    _keep_resident(t, *(s[k] for k in OPERANDS[path]))
    return s


def run(s):
    L, c = xk.lib(), s["case"]
    path, t = c["path"], c.get("type", "d")
    if path == "gemm":
        xk.gemm(OPS[c["op"][0]], OPS[c["op"][1]], 1.5, s["A"], s["B"], c["beta"], s["C"])
        return s["C"]
    if path == "host":
        xk.gemm(xk.NoTrans, xk.NoTrans, 1.5, s["A"], s["B"], 0.0, s["C"])
        xk.invalidate()
        return s["C"]
    if path == "posv":
        X, info, _ = xk.posv_ir(_uplo(c), s["A"], s["B"])
        return {"X": X, "info": info}
    if path == "normal":
        S, X, tr = s["S"], s["X"], c["trans"]
        herm = xk.ConjTrans if t in "cz" else xk.Trans
        form = xk.herk if t in "cz" else xk.syrk
        form(_uplo(c), herm if tr else xk.NoTrans, 1.0, s["G"], 0.0, S, sync=False)
        xk.gemm(herm if tr else xk.NoTrans, xk.NoTrans, 1.0, s["G"], s["Y"], 0.0, X, sync=False)
        xk.potrf(_uplo(c), S, sync=False)
        for op in (xk.NoTrans, herm) if c["uplo"] == "L" else (herm, xk.NoTrans):
            xk.trsm(xk.Left, _uplo(c), op, xk.NonUnit, 1.0, S, X, sync=False)
        _fetch((X, 0))
        return {"X": X, "info": L.xkblas_potrf_info(S.ctypes.data)}
    if path == "sym":
        S, X, B = s["S"], s["X"], s["B"]
        xk.symm(xk.Left, _uplo(c), 1.0, s["A"], B, 0.0, X, sync=False)
        xk.trmm(xk.Left, _uplo(c), xk.NoTrans, xk.NonUnit, 1.0, s["T"], X, sync=False)
        xk.syr2k(_uplo(c), xk.NoTrans, 0.5, X, B, 0.0, S, sync=False)
        _fetch((X, 0), (S, _uplo(c)))
        return {"X": X, "S": S}
    b = s["batch"]
    if c["kept"]:
        L.xkblas_batch_run(b.plan)
    else:
        L.xkblas_batch_run_noalloc(b.problems, b.count)
    L.xkblas_sync()
    return {"C": b.C, "X": b.X}


def _uplo(case):
    return xk.Lower if case["uplo"] == "L" else xk.Upper


def work(case):
    path = case["path"]
    if path == "batch":
        gemms, solves = _shapes(case)
        e, r = SIZE[case["type"]], case["r"]
        return {"bytes": e * (sum(m * k + k * n + 2 * m * n for m, n, k in gemms)
                              + sum(n * (n + 1) // 2 + 2 * n * r for n in solves)),
                "flops": sum(2 * m * n * k for m, n, k in gemms) + sum(n * n * r for n in solves)}
    t = case.get("type", "d")
    e, f = SIZE[t], 4 if t in "cz" else 1
    if path in ("gemm", "host"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": e * (m * k + k * n + m * n * (2 if case.get("beta") else 1)), "flops": f * 2 * m * n * k}
    if path == "normal":
        n, k, r = case["n"], case["k"], case["r"]
        return {"bytes": e * (n * k + k * r + n * r),
                "flops": f * (n * (n + 1) * k + 2 * n * k * r + n * n * n // 3 + 2 * n * n * r)}
    n, r = case["n"], case["r"]
    if path == "posv":
        return {"bytes": e * (n * (n + 1) // 2 + 2 * n * r), "flops": n * n * n // 3 + 2 * n * n * r}
    return {"bytes": e * (3 * n * (n + 1) // 2 + 2 * n * r),
            "flops": f * (2 * n * n * r + n * n * r + 2 * n * (n + 1) * r)}


def _apply(x, op):
    return x if op == "N" else x.T if op == "T" else x.mH


def exact(case, seed):
    path, t = case["path"], case.get("type", "d")
    wide = torch.complex128 if t in "cz" else torch.float64
    if path == "batch":
        b = _Batch(case, seed)
        C, X, r = b.C.double(), b.X.double(), b.r
        for i, (m, n, k) in enumerate(b.gemms):
            A = b.A[int(b.oa[i]):int(b.oa[i]) + m * k].double().view(k, m)
            B = b.B[int(b.ob[i]):int(b.ob[i]) + k * n].double().view(n, k)
            c = C[int(b.oc[i]):int(b.oc[i]) + m * n].view(n, m)
            c.mul_(-0.5).add_(B @ A, alpha=1.5)
        for i, n in enumerate(b.solves):
            T = b.L[int(b.ol[i]):int(b.ol[i]) + n * n].double().view(n, n).T
            v = X[int(b.ox[i]):int(b.ox[i]) + n * r].view(r, n)
            v.copy_(torch.linalg.solve_triangular(T.tril().contiguous(), v.T.contiguous(), upper=False).T)
        return {"C": C.cpu(), "X": X.cpu()}
    x = {k: v.to(wide) for k, v in _inputs(case, seed).items()}
    if path in ("gemm", "host"):
        op = case.get("op", "NN")
        C = 1.5 * (_apply(x["A"], op[0]) @ _apply(x["B"], op[1]))
        if case.get("beta"):
            C += case["beta"] * x["C"]
        return C.cpu().numpy()
    if path == "posv":
        return {"X": _spd_solve(x["A"], x["B"]), "info": None}
    if path == "normal":
        G = x["G"].mH if case["trans"] else x["G"]
        return {"X": _spd_solve(G @ G.mH, G @ x["Y"]), "info": None}
    low = case["uplo"] == "L"
    A, T, B = x["A"], x["T"], x["B"]
    A = A.tril() + A.tril(-1).T if low else A.triu() + A.triu(1).T
    X = (T.tril() if low else T.triu()) @ (A @ B)
    S = X @ B.T
    S = 0.5 * (S + S.T)
    return {"X": X.cpu().numpy(), "S": (S.tril() if low else S.triu()).cpu().numpy()}


def _spd_solve(S, B):
    return torch.cholesky_solve(B.cpu().contiguous(), torch.linalg.cholesky(S.cpu().contiguous())).numpy()
