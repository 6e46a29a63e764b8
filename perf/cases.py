"""Performance cases: the work that programs have utopia_amd do, through its public entry points.

``listed()`` holds the fixed cases, ``draw(rng)`` gives more of the same ranges, ``prepare`` makes what a
program has in hand before the call (operator, plan, solver set up, right-hand sides on the GPU), ``run`` is
one pass, ``work`` what the pass cannot do without, ``exact`` the outputs in 64 bits without this library.

Families (the case's ``path``):

* ``jacobi``   Jacobi-preconditioned CG on the 2D 5-point Laplacian: small systems, bound by latency and launches
* ``mg``       multigrid-preconditioned CG on 3D 7-point operators, FP64 or with the FP32 V-cycle
* ``mprgp``    box-constrained QP (obstacle problem) by MPRGP
* ``pgs``      projected Gauss-Seidel sweeps on the same kind of problem
* ``batched``  many uneven systems with several right-hand sides each, forward and adjoint with gradients
* ``spmv``     one sparse product on matrices without diagonal structure, plain, residual or transposed
* ``galerkin`` the coarse operator P^T A P of a hierarchy's setup
* ``coarse``   dense factorisation and inverse of a coarsest level, and one solve with it
* ``resolve``  a new operator in host memory: multigrid set up from it and one solve (a time or Newton step)
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import utopia_amd as ua
from utopia_amd import autograd as ua_autograd
from utopia_amd import batched as ua_batched

_SHARED = {}


def _context():
    """The program's one context: one stream, as a program that calls the library has it."""
    if "ctx" not in _SHARED:
        _SHARED["ctx"] = ua.Context(0)
    return _SHARED["ctx"]


class _Vector:
    """A torch tensor as the library's vector argument (pointer, length, precision)."""

    def __init__(self, t: torch.Tensor):
        self.t, self.ptr, self.n = t, t.data_ptr(), t.numel()
        self.code = ua.F64 if t.dtype == torch.float64 else ua.F32


class _Owned:
    """A matrix that the library made, freed with the last tensor that views it."""

    def __init__(self, ctx):
        self.ctx, self.m = ctx, ua.uhip_csr()

    def __del__(self):
        ua.lib().uhip_csr_free(self.ctx.h, ctypes.byref(self.m))


class _View:
    def __init__(self, owner, ptr, n, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (int(n),), "typestr": typestr, "data": (int(ptr), False), "version": 2}


def _tensor_of(owner, ptr, n, typestr):
    """Device memory of `owner` as a torch tensor that keeps it alive."""
    return torch.as_tensor(_View(owner, ptr, n, typestr), device="cuda")


def _ref(m):
    return ctypes.byref(m)


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# ------------------------------------------------------------------ cases

def listed():
    return [
        # 2D Poisson, 65,536 rows, rtol 1e-8: the smallest solve that is done in earnest, all latency
        {"name": "cg-jacobi-256x256", "path": "jacobi", "nx": 256, "ny": 256, "rtol": 1e-8},
        # 3D Poisson in FP64, 2.1M rows: an ordinary elliptic solve
        {"name": "mg-cg-fp64-128", "path": "mg", "nx": 128, "ny": 128, "nz": 128, "varcoef": False, "mixed": False,
         "rtol": 1e-10},
        # variable coefficients, 16.8M rows, FP32 V-cycle in FP64 CG: the benchmark's workload, the largest
        {"name": "mg-cg-mixed-256", "path": "mg", "nx": 256, "ny": 256, "nz": 256, "varcoef": True, "mixed": True,
         "rtol": 1e-10},
        # a grid as meshes come, no side a power of two or a multiple of the wavefront
        {"name": "mg-cg-mixed-150x113x90", "path": "mg", "nx": 150, "ny": 113, "nz": 90, "varcoef": True,
         "mixed": True, "rtol": 1e-10},
        # obstacle problem, 1.05M unknowns, to a projected gradient of 1e-9: thousands of short iterations
        {"name": "mprgp-1024x1024", "path": "mprgp", "nx": 1024, "ny": 1024},
        # projected Gauss-Seidel as a smoother-like solver: a fixed number of symmetric multicolour sweeps
        {"name": "pgs-500x300", "path": "pgs", "nx": 500, "ny": 300, "sweeps": 50},
        # 64 uneven systems x 8 right-hand sides, forward solve, adjoint solve and gradients
        {"name": "batched-64x8", "path": "batched", "systems": 64, "lo": 64, "hi": 512, "k": 8, "mixed": True},
        # sparse product with no diagonal structure, FP64 (1M rows of 7, renumbered in blocks)
        {"name": "spmv-renumbered-fp64", "path": "spmv", "kind": "renumbered", "n": 1000000, "f32": False,
         "op": "residual"},
        # ragged graph matrix with empty and very long rows, FP32
        {"name": "spmv-ragged-fp32", "path": "spmv", "kind": "ragged", "n": 300001, "f32": True, "op": "product"},
        # Galerkin product of a 3D fine level, the costly part of a hierarchy's setup
        {"name": "galerkin-96", "path": "galerkin", "nx": 96, "ny": 96, "nz": 96},
        # the dense coarsest level of the largest hierarchy: Cholesky, inverse, one solve
        {"name": "coarse-16x16x16", "path": "coarse", "nx": 16, "ny": 16, "nz": 16},
        # a new operator each step: set up from host arrays and solve
        {"name": "resolve-64x48x40", "path": "resolve", "nx": 64, "ny": 48, "nz": 40, "mixed": True, "rtol": 1e-8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["jacobi", "mg", "mg", "mprgp", "pgs", "batched", "spmv", "spmv", "galerkin", "coarse", "resolve"])
    if path == "jacobi":
        return {"path": path, "nx": _log(rng, 40, 500), "ny": _log(rng, 40, 500), "rtol": 1e-8}
    if path == "mg":
        return {"path": path, "nx": _log(rng, 24, 180), "ny": _log(rng, 24, 180), "nz": _log(rng, 24, 180),
                "varcoef": rng.random() < 0.5, "mixed": rng.random() < 0.5, "rtol": 1e-10}
    if path == "mprgp":
        return {"path": path, "nx": _log(rng, 64, 1000), "ny": _log(rng, 64, 1000)}
    if path == "pgs":
        return {"path": path, "nx": _log(rng, 64, 700), "ny": _log(rng, 64, 700), "sweeps": rng.choice([10, 50])}
    if path == "batched":
        lo = _log(rng, 20, 120)
        return {"path": path, "systems": _log(rng, 4, 48), "lo": lo, "hi": lo * 3, "k": rng.choice([1, 2, 4, 8, 16]),
                "mixed": rng.random() < 0.5}
    if path == "spmv":
        return {"path": path, "kind": rng.choice(["renumbered", "ragged"]), "n": _log(rng, 20000, 1500000),
                "f32": rng.random() < 0.5, "op": rng.choice(["product", "residual", "transpose"])}
    if path == "galerkin":
        return {"path": path, "nx": _log(rng, 12, 96), "ny": _log(rng, 12, 96), "nz": _log(rng, 12, 96)}
    if path == "coarse":
        return {"path": path, "nx": _log(rng, 4, 16), "ny": _log(rng, 4, 16), "nz": _log(rng, 4, 16)}
    return {"path": path, "nx": _log(rng, 16, 64), "ny": _log(rng, 16, 64), "nz": _log(rng, 16, 64),
            "mixed": rng.random() < 0.5, "rtol": 1e-8}


def _levels(dims):
    """Levels of factor-2 coarsening: five (the benchmark's) where the sides allow it, and as many as it
    takes to a coarsest grid of at most 4096 points."""
    levels = 2
    d = [v // 2 for v in dims]
    while (levels < 5 and min(d) >= 8) or math.prod(d) > 4096:
        d = [max(1, v // 2) for v in d]
        levels += 1
    return levels


# ------------------------------------------------------------------ inputs

def _rows(c):
    return c["nx"] * c["ny"] * c.get("nz", 1)


def _stencil3d(c, seed):
    kind = ua.STENCIL_3D7_VARCOEF if c.get("varcoef", True) else ua.STENCIL_3D7
    return ua.gen_stencil(kind, c["nx"], c["ny"], c["nz"], seed=seed)


def _obstacle(c, seed):
    """9-point Laplacian + 1e-3 I, a seeded load, lower bounds -0.05 - 0.15 u (the MPRGP benchmark's problem)."""
    n = _rows(c)
    A = ua.gen_stencil(ua.STENCIL_2D9, c["nx"], c["ny"], shift=1e-3)
    return A, ua.gen_uniform(seed, n), -0.05 - 0.15 * ua.gen_uniform(seed + 1, n, 0, 1)


def _sparse(c, seed):
    """A square matrix with no diagonal structure: a 3D operator renumbered in 64-row blocks, or a graph
    with ragged rows (Pareto lengths up to 3000, some empty, half of the columns near the diagonal)."""
    if c["kind"] == "renumbered":
        s = max(4, round(c["n"] ** (1 / 3)))
        return ua.gen_stencil(ua.STENCIL_3D7_BLOCKPERM, s, s, max(1, c["n"] // (s * s)), seed=seed)
    n, r = c["n"], np.random.RandomState(seed % (1 << 32))
    length = np.minimum(3000, np.floor(4.0 * r.pareto(1.6, n) + 2)).astype(np.int64)
    length[r.random_sample(n) < 0.02] = 0
    row = np.repeat(np.arange(n, dtype=np.int64), length)
    near = np.abs(row + r.randint(-200, 201, row.size)) % n
    col = np.where(r.random_sample(row.size) < 0.5, near, r.randint(0, n, row.size))
    key = np.unique(row * n + col)
    row, col = key // n, (key % n).astype(np.int32)
    rp = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))]).astype(np.int32)
    return ua.Csr(rp, col, r.standard_normal(col.size), (n, n))


def _batch(c, seed):
    """Uneven 2D systems: the sides are the case's own, the edge coefficients the seed's."""
    sides = ua_batched.batch_sides(3, c["systems"], c["lo"], c["hi"])
    return ua_batched.make_batch(sides, seed=1000 * (seed % 1000003), levels=_batch_levels(c))


def _batch_levels(c):
    return max(2, min(ua_batched.levels_for(c["hi"]), int(math.log2(c["lo"] / 3)) + 1))


def prepare(case, seed):
    c, ctx, path = case, _context(), case["path"]
    st = {"case": c, "ctx": ctx}
    if path == "jacobi":
        n = _rows(c)
        A = ua.gen_stencil(ua.STENCIL_2D5, c["nx"], c["ny"])
        b = ua.gen_uniform(seed, n)
        st["solver"] = ua.ConjugateGradient(ctx, "jacobi", atol=c["rtol"] * np.linalg.norm(b), rtol=1e-30, stol=1e-30,
                                            max_it=100000).update(A)
        st["b"], st["x"] = _gpu(b), torch.empty(n, dtype=torch.float64, device="cuda")
    elif path == "mg":
        n = _rows(c)
        A, b = _stencil3d(c, seed), ua.gen_uniform(seed + 100, n)
        ua.srand(1)
        s = ua.ConjugateGradient(ctx, "multigrid_mixed" if c["mixed"] else "multigrid",
                                 atol=c["rtol"] * np.linalg.norm(b), rtol=1e-30, stol=1e-30, max_it=500,
                                 pre_smoothing_steps=2, post_smoothing_steps=2)
        dims = (c["nx"], c["ny"], c["nz"])
        st["solver"] = s.set_transfer_operators(ua.mg_hierarchy(*dims, _levels(dims))).update(A)
        st["b"], st["x"] = _gpu(b), torch.empty(n, dtype=torch.float64, device="cuda")
    elif path in ("mprgp", "pgs"):
        n = _rows(c)
        A, b, lb = _obstacle(c, seed)
        if path == "mprgp":
            s = ua.MPRGP(ctx, atol=1e-9, rtol=0, max_it=1000000)
        else:
            s = ua.ProjectedGaussSeidel(ctx, atol=1e-30, rtol=1e-30, stol=1e-30, max_it=c["sweeps"])
        st["solver"] = s.update(A).set_box_constraints(lb, None)
        st["b"], st["x"] = _gpu(b), torch.empty(n, dtype=torch.float64, device="cuda")
    elif path == "batched":
        p = _batch(c, seed)
        st["op"] = ua_autograd.BatchedSolve(p, c["k"], mixed=c["mixed"], ctx=ctx, rtol=1e-8, max_it=500,
                                            pre_smoothing_steps=2, post_smoothing_steps=2)
        ua.srand(1)
        st["values"] = _gpu(p.A.val).requires_grad_(True)
        st["B"] = _gpu(ua.gen_uniform(seed + 7, p.n * c["k"]).reshape(p.n, c["k"])).requires_grad_(True)
        st["target"] = _gpu(ua.gen_normal(seed + 8, p.n * c["k"]).reshape(p.n, c["k"]))
    elif path == "spmv":
        A, dt = _sparse(c, seed), np.float32 if c["f32"] else np.float64
        n = A.shape[0]
        st["A"] = ua.DeviceCsr(ctx, A, dtype=dt)
        if c["op"] == "transpose":
            ua.check(ua.lib().uhip_csr_plan_transpose(ctx.h, st["A"].ref))
        st["x"] = _Vector(_gpu(ua.gen_uniform(seed + 1, n).astype(dt)))
        st["b"] = _Vector(_gpu(ua.gen_uniform(seed + 2, n).astype(dt)))
        st["y"] = _Vector(torch.empty_like(st["x"].t))
    elif path == "galerkin":
        dims = (c["nx"], c["ny"], c["nz"])
        st["A"] = ua.DeviceCsr(ctx, _stencil3d(c, seed))
        st["P"] = ua.DeviceCsr(ctx, ua.gen_prolongation(*dims))
    elif path == "coarse":
        n = _rows(c)
        st["A"] = ua.DeviceCsr(ctx, _stencil3d(c, seed))
        st["b"] = _gpu(ua.gen_uniform(seed + 1, n))
        st["L"], st["inv"] = (torch.empty(n, n, dtype=torch.float64, device="cuda") for _ in range(2))
        st["x"] = torch.empty_like(st["b"])
    else:
        n, dims = _rows(c), (c["nx"], c["ny"], c["nz"])
        st["A"], st["b"] = _stencil3d(c, seed), ua.gen_uniform(seed + 100, n)
        st["solver"] = ua.ConjugateGradient(ctx, "multigrid_mixed" if c["mixed"] else "multigrid",
                                            atol=c["rtol"] * np.linalg.norm(st["b"]), rtol=1e-30, stol=1e-30,
                                            max_it=500, pre_smoothing_steps=2, post_smoothing_steps=2)
        st["solver"].set_transfer_operators(ua.mg_hierarchy(*dims, _levels(dims)))
    return st


def run(st):
    c, ctx, path, L = st["case"], st["ctx"], st["case"]["path"], ua.lib()
    if path in ("jacobi", "mg", "mprgp", "pgs"):
        x = st["x"]
        ua.check(L.uhip_vec_set_f64(ctx.h, x.numel(), 0.0, _p(x)))  # zero initial guess
        st["solver"].apply_device(_Vector(st["b"]), _Vector(x))
        return x
    if path == "batched":
        X = st["op"](st["values"], st["B"])
        loss = 0.5 * ((X - st["target"]) ** 2).sum()
        grads = torch.autograd.grad(loss, (st["values"], st["B"]))
        return {"X": X.detach(), "values": grads[0], "B": grads[1]}
    if path == "spmv":
        A, x, y = st["A"], st["x"], st["y"]
        if c["op"] == "product":
            A.spmv(x, y)
        elif c["op"] == "residual":
            A.residual(x, st["b"], y)
        else:
            ua.check(L.uhip_spmv_transpose(ctx.h, A.ref, _p(x.t), _p(y.t)))
        return y.t
    if path == "galerkin":
        o = _Owned(ctx)
        ua.check(L.uhip_csr_ptap(ctx.h, st["A"].ref, st["P"].ref, _ref(o.m)), "uhip_csr_ptap")
        return {"rowptr": _tensor_of(o, o.m.rowptr, o.m.nrows + 1, "<i4"), "col": _tensor_of(o, o.m.col, o.m.nnz, "<i4"),
                "val": _tensor_of(o, o.m.val, o.m.nnz, "<f8")}
    if path == "coarse":
        n, info = st["b"].numel(), ctypes.c_int()
        ua.check(L.uhip_csr_to_dense(ctx.h, st["A"].ref, _p(st["L"])))
        ua.check(L.uhip_dense_cholesky(ctx.h, n, _p(st["L"]), n, ctypes.byref(info)))
        ua.check(L.uhip_dense_cholesky_inverse(ctx.h, n, _p(st["L"]), n, _p(st["inv"])))
        ua.check(L.uhip_dense_gemv(ctx.h, n, _p(st["inv"]), _p(st["b"]), ua.F64, _p(st["x"]), ua.F64))
        return {"inverse": st["inv"], "x": st["x"]}
    ua.srand(1)  # the start vectors of the eigenvalue estimates
    return st["solver"].solve(st["A"], st["b"])


# ------------------------------------------------------------------ what a pass cannot do without

def _cg_iteration_bytes(n, diagonals):
    """A p with p.Ap, the residual update, the x and p updates, FP64; the operator is symmetric."""
    return n * ((diagonals + 1) // 2 * 8 + 16 + 24 + 40)


def _vcycle_bytes(n, v):
    """V(2,2): on each level two passes over the (symmetric) operator, nine vector reads or writes;
    7 diagonals on the finest of n rows, 27 below, each level an eighth of the one above."""
    return n * v * (2 * 4 + 9) + n / 7 * v * (2 * 14 + 9)


def _mg_iterations(c):
    """CG iterations to 1e-10: 11 on the Poisson operator, growing with the grid under random coefficients."""
    its = 28 * max(c["nx"], c["ny"], c["nz"]) ** 0.285 if c.get("varcoef", True) else 11
    return its * math.log(c["rtol"]) / math.log(1e-10)


def work(case):
    c, path = case, case["path"]
    if path == "jacobi":
        n, its = _rows(c), 2.3 * max(c["nx"], c["ny"])
        b = its * (_cg_iteration_bytes(n, 5) + 8 * n)
        return {"bytes": b, "flops": its * n * 22}
    if path in ("mg", "resolve"):
        n, its = _rows(c), _mg_iterations(c)
        b = its * (_cg_iteration_bytes(n, 7) + _vcycle_bytes(n, 4 if c["mixed"] else 8))
        if path == "resolve":  # the operator comes from the host: values and columns, read once
            b += 7 * n * 12 + n * 16
        return {"bytes": b, "flops": its * n * 130}
    if path == "mprgp":  # A p; x, g, lb, ub, p, Ap in and x, g, fi out; p and Ap of the next step
        n, its = _rows(c), 2.3 * max(c["nx"], c["ny"])
        return {"bytes": its * n * (5 * 8 + 16 + 9 * 8 + 3 * 8), "flops": its * n * 45}
    if path == "pgs":  # a symmetric sweep reads the operator twice
        n, its = _rows(c), c["sweeps"]
        return {"bytes": its * n * (2 * 5 * 8 + 6 * 8), "flops": its * n * 60}
    if path == "batched":
        mean = (c["hi"] ** 2 - c["lo"] ** 2) / (2 * math.log(c["hi"] / c["lo"]))  # of a log-uniform side's square
        n, k, v, its = c["systems"] * mean, c["k"], 4 if c["mixed"] else 8, 2 * 13
        level = n * (5 * v + 4 * 2 + 9 * k * v) * 4 / 3
        return {"bytes": its * (n * (5 * 8 + k * 8 * 9) + level), "flops": its * n * k * 110}
    if path == "spmv":
        per = 7 if c["kind"] == "renumbered" else 9.8
        v, n = 4 if c["f32"] else 8, c["n"]
        return {"bytes": n * (per * (v + 4) + 4 + v * (3 if c["op"] == "residual" else 2)), "flops": 2 * per * n}
    if path == "galerkin":  # A (7 a row) and P (3.4 a row) in, 27 a coarse row out
        n = _rows(c)
        return {"bytes": n * ((7 + 3.375) * 12 + 8) + n / 8 * (27 * 12 + 4), "flops": n * 2 * (7 * 3.375 + 3.375 * 10)}
    n = _rows(c)  # coarse: n^3/3 for the factor, 2 n^3/3 for the inverse
    return {"bytes": 8.0 * n * n + 8 * 7 * n, "flops": 1.0 * n ** 3}


# ------------------------------------------------------------------ the outputs in 64 bits

def _poisson(b, dims):
    """The Dirichlet Laplacian's solution by sine transforms (dims: x, y[, z]; x runs fastest)."""
    sides = [d for d in dims if d > 1]
    t = np.asarray(b, np.float64).reshape(sides[::-1])
    eig = 0.0
    basis = []
    for axis, d in enumerate(sides[::-1]):
        k = np.arange(1, d + 1)
        basis.append(math.sqrt(2.0 / (d + 1)) * np.sin(np.pi * np.outer(k, k) / (d + 1)))
        shape = [1] * len(sides)
        shape[axis] = d
        eig = eig + (2 - 2 * np.cos(np.pi * k / (d + 1))).reshape(shape)

    def transform(u):
        for axis, s in enumerate(basis):
            u = np.moveaxis(np.tensordot(s, u, axes=(1, axis)), 0, axis)
        return u

    return transform(transform(t) / eig).reshape(-1)


def _rows_of(rowptr):
    return np.repeat(np.arange(rowptr.size - 1, dtype=np.int64), np.diff(rowptr))


def _sum_by_key(key, val):
    """Sorted distinct keys and the sum of the values of each."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    key, order = torch.sort(torch.from_numpy(key).to(dev), stable=True)
    val = torch.from_numpy(val).to(dev)[order]
    distinct, where = torch.unique_consecutive(key, return_inverse=True)
    total = torch.zeros(distinct.numel(), dtype=torch.float64, device=dev).index_add_(0, where, val)
    return distinct.cpu().numpy(), total.cpu().numpy()


def _product(ar, ac, av, brp, bc, bv, ncols):
    """Rows, columns and values of A B, A given by entries and B by CSR arrays."""
    length = np.diff(brp)[ac]
    start = np.repeat(brp[ac].astype(np.int64) - np.concatenate([[0], np.cumsum(length)[:-1]]), length)
    e = start + np.arange(int(length.sum()))
    key, val = _sum_by_key(np.repeat(ar, length) * ncols + bc[e], np.repeat(av, length) * bv[e])
    return key // ncols, key % ncols, val


def exact(case, seed):
    c, path = case, case["path"]
    if path == "jacobi":
        return _poisson(ua.gen_uniform(seed, _rows(c)), (c["nx"], c["ny"]))
    if path == "mg" and not c["varcoef"]:
        return _poisson(ua.gen_uniform(seed + 100, _rows(c)), (c["nx"], c["ny"], c["nz"]))
    if path == "spmv":
        A, dt = _sparse(c, seed), np.float32 if c["f32"] else np.float64
        n = A.shape[0]
        val = A.val.astype(dt).astype(np.float64)
        x, b = (ua.gen_uniform(seed + k, n).astype(dt).astype(np.float64) for k in (1, 2))
        row, col = _rows_of(A.rowptr), A.col[:A.nnz]
        if c["op"] == "transpose":
            return np.bincount(col, weights=val * x[row], minlength=n)
        y = np.bincount(row, weights=val * x[col], minlength=n)
        return b - y if c["op"] == "residual" else y
    if path == "galerkin":
        A, P = _stencil3d(c, seed), ua.gen_prolongation(c["nx"], c["ny"], c["nz"])
        m, prow = P.shape[1], _rows_of(P.rowptr)
        r, k, v = _product(_rows_of(A.rowptr), A.col, A.val, P.rowptr, P.col, P.val, m)
        rp = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=A.shape[0]))])
        order = np.lexsort((prow, P.col))  # the entries of P^T
        r, k, v = _product(P.col[order].astype(np.int64), prow[order], P.val[order], rp, k, v, m)
        return {"rowptr": None, "col": None, "val": v}
    if path == "coarse":
        A, n = _stencil3d(c, seed), _rows(c)
        dense = torch.zeros(n, n, dtype=torch.float64)
        dense[torch.from_numpy(_rows_of(A.rowptr)), torch.from_numpy(A.col.astype(np.int64))] = torch.from_numpy(A.val)
        if torch.cuda.is_available():
            dense = dense.cuda()
        inv = torch.cholesky_inverse(torch.linalg.cholesky(dense))
        return {"inverse": inv, "x": inv @ torch.from_numpy(ua.gen_uniform(seed + 1, n)).to(inv.device)}
    return None
