"""Workloads whose speed this library is judged by.

Each case is one pass through the public entry points (linalglib_amd.lal and
linalglib_amd.torch_solve) as a program on top of them would make it: the
sparse products, one step of a hand-written CG, the hierarchy build, the
preconditioner, the solvers in FP64 and mixed precision, and the
differentiable solve.  `listed()` names fixed sizes, `draw()` picks others of
the same ranges.  Matrices are this package's own generators (Poisson and
log-normal diffusion grids, kNN graph Laplacians).
"""
import ctypes as C

import numpy as np
import torch

from linalglib_amd import lal, problems
from linalglib_amd.torch_solve import saamg_solve

DEV = "cuda"


def listed():
    return [
        # One CG step written by the caller on the BLAS-level entry points (a
        # LinAlgLib program whose device shims call this library): SpMV, two
        # inner products read back, three vector updates, small vectors.
        {"name": "cg_step_2d_128", "kind": "cg_step", "op": "poisson2d", "nx": 128, "ny": 128},
        # The metric's own SpMV: 7-point Poisson 128^3 in FP64, caller's matrix.
        {"name": "spmv_f64_poisson_128", "kind": "spmv", "op": "poisson3d", "dtype": "f64",
         "nx": 128, "ny": 128, "nz": 128},
        # FP32 SpMV on a box with odd sides (ragged last blocks).
        {"name": "spmv_f32_poisson_box", "kind": "spmv", "op": "poisson3d", "dtype": "f32",
         "nx": 161, "ny": 97, "nz": 113},
        # Residual of an irregular graph operator (12-20 entries per row).
        {"name": "residual_f64_knn_150k", "kind": "residual", "op": "knn", "dtype": "f64",
         "n": 150001},
        # C = A A on an irregular graph: both passes of the sparse product.
        {"name": "spgemm_knn_60k", "kind": "spgemm", "op": "knn", "n": 60000},
        # Hierarchy build and its first application, small: what a caller pays
        # whenever the values of a small operator change.
        {"name": "setup_diffusion_25", "kind": "setup", "op": "diffusion", "nx": 25,
         "sigma": 1.0, "f32": False},
        # Hierarchy build near the headline's size, with the FP32 levels.
        {"name": "setup_diffusion_121", "kind": "setup", "op": "diffusion", "nx": 121,
         "sigma": 1.0, "f32": True},
        # One preconditioner application (V(1,1), FP64) on log-normal diffusion:
        # what an outer solver of the caller's own pays per iteration.
        {"name": "vcycle_diffusion_97", "kind": "vcycle", "op": "diffusion", "nx": 97,
         "sigma": 1.5},
        # Whole small solve, latency bound.
        {"name": "pcg_poisson2d_128", "kind": "pcg", "op": "poisson2d", "nx": 128, "ny": 128,
         "tol": 1e-8},
        # Whole FP64 solve on log-normal diffusion.
        {"name": "pcg_diffusion_101", "kind": "pcg", "op": "diffusion", "nx": 101, "sigma": 1.5,
         "tol": 1e-10},
        # The headline: mixed-precision solve of 3D Poisson 128^3 to 1e-10.
        {"name": "pcg_reliable_poisson_128", "kind": "pcg_reliable", "op": "poisson3d",
         "nx": 128, "ny": 128, "nz": 128, "tol": 1e-10},
        # Differentiable solve, forward and backward, hierarchy built per call:
        # one step of an inverse problem for face conductances.
        {"name": "gradient_faces_64", "kind": "gradient", "op": "faces", "nx": 64,
         "sigma": 1.0, "tol": 1e-11},
    ]


def _log_int(rng, lo, hi):
    return int(round(np.exp(rng.uniform(np.log(lo), np.log(hi)))))


def draw(rng):
    kind = rng.choice(["cg_step", "spmv", "residual", "spgemm", "setup", "vcycle", "pcg",
                       "pcg_reliable", "gradient"])
    c = {"kind": kind}
    if kind == "gradient":
        c.update(op="faces", nx=_log_int(rng, 16, 64), sigma=round(rng.uniform(0.3, 1.0), 3),
                 tol=1e-11)
        return c
    ops = {"cg_step": ["poisson2d", "poisson3d"], "spgemm": ["knn", "diffusion"],
           "setup": ["knn", "diffusion"]}  # products and setups take seeded values
    c["op"] = rng.choice(ops.get(kind, ["poisson2d", "poisson3d", "diffusion", "knn"]))
    big = kind != "cg_step"
    if c["op"] == "poisson2d":
        c.update(nx=_log_int(rng, 40, 700 if big else 160),
                 ny=_log_int(rng, 40, 700 if big else 160))
    elif c["op"] == "poisson3d":
        top = 128 if big else 29
        c.update(nx=_log_int(rng, 12, top), ny=_log_int(rng, 12, top), nz=_log_int(rng, 12, top))
    elif c["op"] == "diffusion":
        c.update(nx=_log_int(rng, 16, 71 if kind == "spgemm" else 101), sigma=round(rng.uniform(0.3, 1.5), 3))
    else:
        c["n"] = _log_int(rng, 3000, 60000 if kind == "spgemm" else 150001)
    if kind in ("spmv", "residual"):
        c["dtype"] = rng.choice(["f64", "f32"])
    elif kind == "setup":
        c["f32"] = rng.choice([False, True])
    elif kind in ("pcg", "pcg_reliable"):
        c["tol"] = rng.choice([1e-8, 1e-10])
    return c


# ---------------------------------------------------------------- the inputs
def _matrix(case, seed):
    """(row_ptr, col_ind, val, m) in numpy; values from the seed where the
    operator has coefficients."""
    rng = np.random.default_rng([seed, 11])
    op = case["op"]
    if op == "poisson2d":
        return problems.poisson2d(case["nx"], case["ny"])
    if op == "poisson3d":
        return problems.poisson3d(case["nx"], case["ny"], case["nz"])
    if op == "diffusion":
        n = case["nx"]
        return problems.diffusion3d(n, cell_kappa=np.exp(case["sigma"] *
                                                         rng.standard_normal((n, n, n))))
    # the graph belongs to the case, its edge weights to the seed
    rp, ci, m, edges, entry, edge, sign, dpos = problems.knn_laplacian(case["n"], seed=7)
    w = np.exp(0.5 * rng.standard_normal(len(edges)))
    val = np.bincount(entry, weights=sign * w[edge], minlength=len(ci))
    val[dpos] += 1e-2
    return rp, ci, val, m


def _faces(case, seed):
    rng = np.random.default_rng([seed, 12])
    rp, ci, m, nf, entry, face, sign = problems.diffusion_faces(case["nx"])
    k = np.exp(case["sigma"] * rng.standard_normal(nf))
    return rp, ci, np.bincount(entry, weights=sign * k[face], minlength=len(ci)), m


def _vec(m, seed, which):
    return np.random.default_rng([seed, which]).uniform(-1.0, 1.0, m)


def _host_inputs(case, seed):
    """The matrix and vectors of one case on the host (numpy, FP64 or the
    case's FP32)."""
    rp, ci, v, m = _faces(case, seed) if case["op"] == "faces" else _matrix(case, seed)
    x, b = _vec(m, seed, 1), _vec(m, seed, 2)
    if case.get("dtype") == "f32":
        v, x, b = v.astype(np.float32), x.astype(np.float32), b.astype(np.float32)
    return rp, ci, v, m, x, b


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def prepare(case, seed):
    rp, ci, v, m, x, b = _host_inputs(case, seed)
    kind = case["kind"]
    s = {"kind": kind, "m": m, "nnz": len(ci), "rp": _dev(rp), "ci": _dev(ci), "v": _dev(v),
         "tol": case.get("tol")}
    if kind in ("pcg", "pcg_reliable"):
        # a right-hand side with a known solution
        s["b"] = _dev(problems.rhs_from_solution(rp, ci, v, x))
    elif kind == "gradient":
        s["b"] = _dev(problems.rhs_from_solution(rp, ci, v, x)).requires_grad_(True)
        s["v"].requires_grad_(True)
        s["g"] = _dev(problems.rhs_from_solution(rp, ci, v, b))  # dL/dx of the loss above
        return s
    else:
        s["x"], s["b"] = _dev(x), _dev(b)
    s["h"] = lal.Handle()
    if kind in ("spmv", "residual", "cg_step"):
        s["d"] = lal.CsrDescr(s["h"], m, m, s["nnz"], s["rp"], s["ci"])
        s["y"] = torch.empty_like(s["x"])
    if kind == "cg_step":
        s["f"] = C.c_double()
    elif kind == "setup":
        s["f32"] = int(case["f32"])
        s["y"] = torch.empty_like(s["b"])
    elif kind in ("vcycle", "pcg", "pcg_reliable"):
        s["H"] = lal.Hierarchy(s["h"], m, s["nnz"], s["rp"], s["ci"], s["v"],
                               build_f32=int(kind == "pcg_reliable"))
        s["y"] = torch.empty(m, dtype=torch.float64, device=DEV)
    return s


# ------------------------------------------------------------------ the pass
def _cg_step(s):
    """x, r, p of one CG step from x = 0, r = p = b (cg.cpp's order)."""
    h, m, f, ptr, call = s["h"].h, s["m"], s["f"], lal.ptr, lal.call
    x, r, p, q = torch.zeros_like(s["b"]), s["b"].clone(), s["x"].clone(), s["y"]
    call("lal_csrmv_f64", h, s["d"].d, m, m, s["nnz"], 1.0, ptr(s["rp"]), ptr(s["ci"]),
         ptr(s["v"]), ptr(p), 0.0, ptr(q))
    call("lal_dot_f64", h, m, ptr(r), ptr(r), C.byref(f))
    gamma = f.value
    call("lal_dot_f64", h, m, ptr(q), ptr(p), C.byref(f))
    alpha = gamma / f.value
    call("lal_axpy_f64", h, m, alpha, ptr(p), ptr(x))
    call("lal_axpy_dot_f64", h, m, -alpha, ptr(q), ptr(r), ptr(r), C.byref(f))
    beta = f.value / gamma
    call("lal_axpby_f64", h, m, 1.0, ptr(r), beta, ptr(p))
    call("lal_norm_inf_f64", h, m, ptr(r), C.byref(f))
    return {"x": x, "r": r, "p": p, "q": q, "alpha": alpha, "beta": beta, "norm": f.value}


def run(s):
    kind, ptr, call = s["kind"], lal.ptr, lal.call
    if kind == "spmv":
        fn = "lal_csrmv_f64" if s["v"].dtype == torch.float64 else "lal_csrmv_f32"
        call(fn, s["h"].h, s["d"].d, s["m"], s["m"], s["nnz"], 1.0, ptr(s["rp"]), ptr(s["ci"]),
             ptr(s["v"]), ptr(s["x"]), 0.0, ptr(s["y"]))
        return s["y"]
    if kind == "residual":
        fn = "lal_residual_f64" if s["v"].dtype == torch.float64 else "lal_residual_f32"
        call(fn, s["h"].h, s["d"].d, s["m"], s["m"], s["nnz"], ptr(s["rp"]), ptr(s["ci"]),
             ptr(s["v"]), ptr(s["x"]), ptr(s["b"]), ptr(s["y"]))
        return s["y"]
    if kind == "cg_step":
        return _cg_step(s)
    if kind == "spgemm":
        m, nnz, h = s["m"], s["nnz"], s["h"].h
        crp = torch.empty(m + 1, dtype=torch.int32, device=DEV)
        n = C.c_int()
        call("lal_csrgemm_nnz", h, m, m, m, nnz, ptr(s["rp"]), ptr(s["ci"]), nnz, ptr(s["rp"]),
             ptr(s["ci"]), ptr(crp), C.byref(n))
        cci = torch.empty(n.value, dtype=torch.int32, device=DEV)
        cv = torch.empty(n.value, dtype=torch.float64, device=DEV)
        call("lal_csrgemm_solve_f64", h, m, m, m, nnz, ptr(s["rp"]), ptr(s["ci"]), ptr(s["v"]),
             nnz, ptr(s["rp"]), ptr(s["ci"]), ptr(s["v"]), ptr(crp), ptr(cci), ptr(cv))
        return {"rp": crp, "ci": cci, "v": cv}
    if kind == "setup":
        H = lal.Hierarchy(s["h"], s["m"], s["nnz"], s["rp"], s["ci"], s["v"],
                          build_f32=s["f32"])
        H.precond(s["b"], s["y"])
        return s["y"]
    if kind == "vcycle":
        s["H"].precond(s["b"], s["y"])
        return s["y"]
    if kind == "gradient":
        x = saamg_solve(s["v"], s["b"], s["rp"], s["ci"], tol=s["tol"])
        dv, db = torch.autograd.grad(x, (s["v"], s["b"]), s["g"])
        return {"x": x.detach(), "dv": dv, "db": db}
    s["y"].zero_()
    solve = s["H"].pcg if kind == "pcg" else s["H"].pcg_reliable
    info = solve(s["b"], s["y"], rel_tol=s["tol"], abs_tol=1e-300, max_iter=500)
    if not info.converged:
        raise RuntimeError("solve did not converge")
    return s["y"]


# ------------------------------------------------------ sizes and references
def _counts(case):
    """(rows, nonzeros) of the case's matrix (kNN: the mean row length)."""
    op = case["op"]
    if op == "knn":
        return case["n"], int(case["n"] * 14.8)
    if op == "poisson2d":
        nx, ny = case["nx"], case["ny"]
        return nx * ny, 5 * nx * ny - 2 * (nx + ny)
    nx = case["nx"]
    ny, nz = case.get("ny", nx), case.get("nz", nx)
    return nx * ny * nz, 7 * nx * ny * nz - 2 * (nx * ny + ny * nz + nx * nz)


# V-cycle applications of a solve, roughly: what convergence to the case's
# tolerance takes on each operator with this preconditioner
_ITERATIONS = {"poisson2d": 36, "poisson3d": 32, "diffusion": 56, "knn": 45, "faces": 60}


def work(case):
    m, nnz = _counts(case)
    kind = case["kind"]
    e = 4 if case.get("dtype") == "f32" or kind == "pcg_reliable" else 8
    matrix = nnz * (e + 4) + 4 * (m + 1)
    # a hierarchy of these operators holds about 2.7 times the finest
    # operator's entries, its transfer operators about 0.8 times
    cycle = {"bytes": 2.7 * matrix + 0.8 * nnz * (e + 4) + 3 * e * m, "flops": 2 * 3.5 * nnz}
    if kind == "spmv":
        return {"bytes": matrix + 2 * e * m, "flops": 2 * nnz}
    if kind == "residual":
        return {"bytes": matrix + 3 * e * m, "flops": 2 * nnz}
    if kind == "cg_step":
        return {"bytes": matrix + 7 * 8 * m, "flops": 2 * nnz + 12 * m}
    if kind == "spgemm":
        grow = 4.1 if case["op"] == "knn" else 3.5  # nonzeros of A A per nonzero of A
        per_row = nnz / m
        return {"bytes": 2 * (12 * nnz + 4 * m) + 12 * grow * nnz + 4 * m,
                "flops": 2 * per_row * nnz}
    if kind == "setup":
        extra = 4 * 3.5 * nnz if case["f32"] else 0
        return {"bytes": 12 * nnz + 12 * 3.5 * nnz + extra + cycle["bytes"],
                "flops": 2 * 20 * nnz + cycle["flops"]}
    if kind == "vcycle":
        return cycle
    its = _ITERATIONS[case["op"]]
    solve = {"bytes": its * (cycle["bytes"] + matrix + 8 * e * m),
             "flops": its * (cycle["flops"] + 2 * nnz + 10 * m)}
    if kind == "gradient":
        return {"bytes": 2 * solve["bytes"] + 12 * 3.5 * nnz + 8 * nnz,
                "flops": 2 * solve["flops"] + 2 * 20 * nnz}
    return solve


def _product(rp, ci, v, x, m):
    rows = np.repeat(np.arange(m), np.diff(rp))
    return np.bincount(rows, weights=v.astype(np.float64) * x.astype(np.float64)[ci], minlength=m)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("setup", "vcycle"):
        return None  # defined by the hierarchy's own rounding-dependent patterns
    rp, ci, v, m, x, b = _host_inputs(case, seed)
    if kind == "spmv":
        return _product(rp, ci, v, x, m)
    if kind == "residual":
        return b.astype(np.float64) - _product(rp, ci, v, x, m)
    if kind == "cg_step":
        q = _product(rp, ci, v, x, m)
        gamma = float(b @ b)
        alpha = gamma / float(q @ x)
        r = b - alpha * q
        beta = float(r @ r) / gamma
        return {"x": alpha * x, "r": r, "p": r + beta * x, "q": q, "alpha": alpha, "beta": beta,
                "norm": float(np.abs(r).max())}
    if kind == "spgemm":
        # every product a_ik a_kj, summed per (i, j)
        lens = np.diff(rp)
        rows = np.repeat(np.arange(m), lens)
        reps = lens[ci]
        first = np.cumsum(reps) - reps
        at = np.arange(int(reps.sum())) - np.repeat(first, reps) + np.repeat(rp[ci], reps)
        key = np.repeat(rows, reps).astype(np.int64) * m + ci[at]
        prod = np.repeat(v, reps) * v[at]
        keys, inv = np.unique(key, return_inverse=True)
        val = np.bincount(inv, weights=prod)
        crp = np.zeros(m + 1, np.int64)
        np.cumsum(np.bincount(keys // m, minlength=m), out=crp[1:])
        return {"rp": crp.astype(np.int32), "ci": (keys % m).astype(np.int32), "v": val}
    if kind == "gradient":
        rows = np.repeat(np.arange(m), np.diff(rp))
        return {"x": x, "dv": -b[rows] * x[ci], "db": b}
    return x  # the right-hand side was made from it
