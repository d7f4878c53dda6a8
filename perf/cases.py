"""The measured work of the preconditioned-Krylov path: single products, whole
solves with each preconditioner family, the batched differentiable solve, all
through the public Python classes, from about a thousand rows to millions.

Every system is built as b = A x_true from a seeded x_true, so x_true is the
exact answer of a solve; a solve stops at the reference's default criterion
(relative residual 1e-8).
"""
import math

import numpy as np
import torch

import prispack_amd as pp
from prispack_amd import autograd as ppg

TOL = 1e-8

# kinds of drawn cases and how often each is drawn
_KINDS = ["products", "cg_ict_2d", "cg_ict_2d", "cg_ict_3d", "cg_ildlt_2d", "gmres_ilut", "cg_ic0", "cg_ic0",
          "gmres_ilu0", "new_values", "multilevel", "batch"]


def listed():
    return [
        # an outer iteration of the caller's own: y = A x, z = A^T y, r = b - A x on a small
        # 2D operator; the smallest call, launch and host latency
        {"name": "products_small_f64", "kind": "products", "nx": 48, "ny": 41, "nz": 1, "beta": 20.0,
         "dtype": "f64"},
        # the same in FP32 on a ragged 3D operator
        {"name": "products_3d_f32", "kind": "products", "nx": 127, "ny": 97, "nz": 61, "beta": 20.0,
         "dtype": "f32"},
        # the reference's default solver on a small grid: FlexibleCG + threshold Cholesky
        {"name": "cg_ict_small", "kind": "cg_ict", "nx": 37, "ny": 31, "nz": 1, "tau": 1e-3},
        # the reference's own test workload, 2D Poisson 128^2
        {"name": "cg_ict_2d", "kind": "cg_ict", "nx": 128, "ny": 128, "nz": 1, "tau": 1e-3},
        # the same method on the 64^3 Poisson problem, whose factor is one connected part
        {"name": "cg_ict_3d", "kind": "cg_ict", "nx": 64, "ny": 64, "nz": 64, "tau": 1e-2},
        # the reference's nonsymmetric default: FGMRES(30) + ILUT(20, 1e-2), convection-diffusion, ragged
        {"name": "gmres_ilut_3d", "kind": "gmres_ilut", "nx": 50, "ny": 43, "nz": 31, "beta": 20.0, "lfil": 20,
         "tau": 1e-2, "precision": "fp64"},
        # large SPD systems: colour-ordered IC(0), full FP64 and mixed precision
        {"name": "cg_ic0_128_fp64", "kind": "cg_ic0", "nx": 128, "ny": 128, "nz": 128, "precision": "fp64"},
        {"name": "cg_ic0_128_mixed", "kind": "cg_ic0", "nx": 128, "ny": 128, "nz": 128, "precision": "mixed"},
        # large nonsymmetric systems: colour-ordered ILU(0) + FGMRES(30)
        {"name": "gmres_ilu0_100", "kind": "gmres_ilu0", "nx": 100, "ny": 100, "nz": 100, "beta": 20.0,
         "precision": "fp64"},
        # a time step: new coefficients on a known pattern, numeric factorization, mixed solve
        {"name": "new_values_3d", "kind": "new_values", "nx": 81, "ny": 72, "nz": 65, "precision": "mixed"},
        # the reference's multilevel low-rank preconditioner
        {"name": "amsed_64", "kind": "amsed", "nx": 64, "ny": 64, "nz": 64, "precision": "fp64"},
        # a training step through 256 uneven variable-coefficient systems: solve, adjoint solve, gradients
        {"name": "batch_256", "kind": "batch", "systems": 256, "side0": 32, "side1": 256, "precision": "mixed"},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi):
    """A 3D grid of lo^3 to hi^3 points, the count spread over its logarithm,
    the sides uneven."""
    s = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    a, b = math.exp(rng.uniform(-0.25, 0.25)), math.exp(rng.uniform(-0.25, 0.25))
    nx, ny = max(4, round(s * a)), max(4, round(s * b))
    return {"nx": nx, "ny": ny, "nz": min(max(4, round(s / (a * b))), hi ** 3 // (nx * ny))}


def _rect(rng, lo, hi):
    s = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    a = math.exp(rng.uniform(-0.35, 0.35))
    nx = max(4, round(s * a))
    return {"nx": nx, "ny": min(max(4, round(s / a)), hi * hi // nx), "nz": 1}


def draw(rng):
    kind = rng.choice(_KINDS)
    prec = rng.choice(["fp64", "mixed"])
    if kind == "products":
        dims = _box(rng, 10, 110) if rng.random() < 0.6 else _rect(rng, 24, 1000)
        return {"kind": kind, **dims, "beta": 20.0, "dtype": rng.choice(["f64", "f32"])}
    if kind == "cg_ict_2d":
        return {"kind": "cg_ict", **_rect(rng, 24, 160), "tau": rng.choice([1e-3, 3e-3, 1e-2])}
    if kind == "cg_ict_3d":
        return {"kind": "cg_ict", **_box(rng, 10, 60), "tau": rng.choice([3e-3, 1e-2])}
    if kind == "cg_ildlt_2d":
        return {"kind": "cg_ildlt", **_rect(rng, 24, 128), "tau": rng.choice([1e-3, 1e-2])}
    if kind == "gmres_ilut":
        return {"kind": kind, **_box(rng, 10, 40), "beta": 20.0, "lfil": rng.choice([5, 10, 20]), "tau": 1e-2,
                "precision": prec}
    if kind == "cg_ic0":
        dims = _box(rng, 24, 120) if rng.random() < 0.7 else _rect(rng, 100, 700)
        return {"kind": kind, **dims, "precision": prec}
    if kind == "gmres_ilu0":
        return {"kind": kind, **_box(rng, 24, 90), "beta": 20.0, "precision": prec}
    if kind == "new_values":
        return {"kind": kind, **_box(rng, 34, 80), "precision": prec}
    if kind == "multilevel":
        return {"kind": rng.choice(["amsed", "gmslr"]), **_box(rng, 24, 56), "beta": 20.0, "precision": prec}
    prec = rng.choice(["mixed", "mixed", "fp64"])
    s1 = _logint(rng, 48, 224 if prec == "mixed" else 112)
    return {"kind": "batch", "systems": _logint(rng, 16, 200), "side0": max(16, s1 // rng.randint(2, 6)),
            "side1": s1, "precision": prec}


# ----------------------------------------------------------------------------- inputs
def _matrix(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["kind"] in ("products", "gmres_ilut", "gmres_ilu0", "gmslr"):
        b = case["beta"]
        return pp.generate_upwind(nx, ny, nz, b, b / 2, b / 4)
    return pp.generateLaplacianCSR(nx, ny, nz)


def _csr_times(A, x):
    rp, ci, v = A
    return np.add.reduceat(v * x[ci], rp[:-1].astype(np.int64))


def _truth(n, seed, which=0):
    return np.random.default_rng([seed, which]).standard_normal(n)


def _row_scale(n, seed):
    # log-normal row and column scaling of the new values: D A D keeps the pattern and stays SPD
    return np.exp(0.3 * np.random.default_rng([seed, 7]).standard_normal(n))


def _batch_sides(case):
    # the sizes are the batch's own; the coefficients and right-hand sides come from the seed
    r = np.random.default_rng([case["systems"], case["side0"], case["side1"]])
    return r.integers(case["side0"], case["side1"] + 1, case["systems"]).tolist()


def _batch_kappa(side, i, seed):
    return np.exp(np.random.default_rng([seed, 100 + i]).standard_normal(side * side))


def _batch_systems(case, seed):
    return [pp.generate_vardiff2d(s, _batch_kappa(s, i, seed)) for i, s in enumerate(_batch_sides(case))]


def _joined(systems):
    """Block-diagonal CSR of the systems."""
    rps, cis, row, nnz = [np.zeros(1, np.int64)], [], 0, 0
    for rp, ci, _ in systems:
        rps.append(rp[1:].astype(np.int64) + nnz)
        cis.append(ci.astype(np.int64) + row)
        row += len(rp) - 1
        nnz += int(rp[-1])
    return np.concatenate(rps), np.concatenate(cis), np.concatenate([s[2] for s in systems])


def _cuda(a, dtype=torch.float64):
    return torch.tensor(a, dtype=dtype, device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        systems = _batch_systems(case, seed)
        J = _joined(systems)
        n = len(J[0]) - 1
        B = pp.BatchedSystems(systems, ordering=1)
        B.tune()
        return {"case": case, "batch": B, "values": _cuda(J[2]).requires_grad_(),
                "b": _cuda(_csr_times(J, _truth(n, seed))).requires_grad_(),
                "gx": _cuda(_csr_times(J, _truth(n, seed, 1)))}
    A = _matrix(case)
    n = len(A[0]) - 1
    M = pp.CSRMatrix(*A)
    st = {"case": case, "A": M, "n": n}
    if kind == "products":
        dt = torch.float64 if case["dtype"] == "f64" else torch.float32
        st["x"] = _cuda(_truth(n, seed), dt)
        st["b"] = _cuda(_truth(n, seed, 1), dt)
        st["y"], st["z"] = torch.zeros_like(st["x"]), torch.zeros_like(st["x"])
        return st
    f32 = case.get("precision") == "mixed"
    if kind == "new_values":
        rp, ci, v = A
        d = _row_scale(n, seed)
        rows = np.repeat(np.arange(n), np.diff(rp.astype(np.int64)))
        st["P"] = pp.IC0(M, make_f32=f32, ordering=1)
        st["P"].setup()  # on the values of the step before
        A = (rp, ci, d[rows] * v * d[ci])
        st["values"] = _cuda(A[2])
    elif kind == "cg_ict":
        st["P"] = pp.IncompleteCholesky(M, case["tau"])
    elif kind == "cg_ildlt":
        st["P"] = pp.IncompleteLDLT(M, case["tau"])
    elif kind == "gmres_ilut":
        st["P"] = pp.IncompleteLU(M, case["lfil"], case["tau"], make_f32=f32)
    elif kind == "cg_ic0":
        st["P"] = pp.IC0(M, make_f32=f32, ordering=1)
    elif kind == "gmres_ilu0":
        st["P"] = pp.ILU0(M, make_f32=f32, ordering=1)
    else:
        st["P"] = (pp.AMSED if kind == "amsed" else pp.GMSLR)(M, levels=3, ndom=16, rank=32)
    if kind != "new_values":
        st["P"].setup()
    st["b"] = _cuda(_csr_times(A, _truth(n, seed)))
    return st


# ----------------------------------------------------------------------------- one pass
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "batch":
        values, b = st["values"], st["b"]
        values.grad = b.grad = None
        x = ppg.batched_solve(values, b, st["batch"], precision=case["precision"], tol=TOL)
        x.backward(st["gx"])
        return {"x": x.detach(), "grad_values": values.grad, "grad_b": b.grad}
    A = st["A"]
    if kind == "products":
        A.MatPVec(st["x"], st["y"])
        A.transMatPVec(st["y"], st["z"], alpha=1.0, beta=0.0)
        r = st["b"].clone()
        A.MatPVec(st["x"], r, alpha=-1.0, beta=1.0)
        return {"y": st["y"], "z": st["z"], "r": r}
    if kind == "new_values":
        A.set_values(st["values"])
        st["P"].refactor()
    precision = case.get("precision", "fp64")
    if kind in ("gmres_ilut", "gmres_ilu0", "gmslr"):
        solver = pp.GMRES(st["n"], st["P"], TOL, pp.FlexibleGMRES, maxIter=3000, precision=precision)
        solver.setRestart(True, 30)
    else:
        solver = pp.CG(st["n"], st["P"], pp.FlexibleCG, tol=TOL, maxIter=2000, precision=precision)
    x = torch.zeros(st["n"], dtype=torch.float64, device="cuda")
    solver.solve(A, st["b"], x)
    return x


# ----------------------------------------------------------------------------- what a pass needs
def _iterations(case):
    """About how many iterations the method takes (measured at the listed
    sizes; CG grows with the grid's side, and the restarted GMRES too)."""
    s = max(case["nx"], case["ny"], case["nz"])
    kind = case["kind"]
    if kind in ("cg_ict", "cg_ildlt"):
        per_side = (0.15 if case["nz"] == 1 else 0.3) * (case["tau"] / 1e-3) ** 0.35
        return 3 + per_side * s
    if kind == "gmres_ilut":
        return 5 + 0.4 * s
    if kind == "gmres_ilu0":
        return 1.7 * s
    if kind in ("amsed", "gmslr"):
        return 5 + 0.5 * s
    return (1.5 if case["nz"] == 1 else 1.3) * s  # colour-ordered IC(0)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        m = (case["side0"] + case["side1"]) / 2
        rows = case["systems"] * (case["side0"] ** 2 + case["side0"] * case["side1"] + case["side1"] ** 2) / 3
        entry = 4 if case["precision"] == "mixed" else 8
        iters = 2 * 2.6 * m  # solve and adjoint solve
        # per iteration the operator's values and the factor's once, x, r, p read and written
        return {"bytes": rows * (iters * entry * (5 + 3 + 6) + 8 * (5 + 5 + 5)), "flops": rows * iters * 2 * (10 + 5)}
    n = case["nx"] * case["ny"] * case["nz"]
    per_row = 5 if case["nz"] == 1 else 7
    if kind == "products":
        e = 8 if case["dtype"] == "f64" else 4
        # three products: the values, columns and row pointers once each, inputs and outputs
        return {"bytes": 3 * n * (per_row * (e + 4) + 4) + 7 * n * e, "flops": 3 * 2 * n * per_row}
    e = 4 if case.get("precision") == "mixed" else 8
    fill = 1.0
    if kind in ("cg_ict", "cg_ildlt", "gmres_ilut", "amsed", "gmslr"):
        fill = 2.5
    # an iteration reads the matrix's values and the factor's once (indices
    # aside: a stencil's can be told from its rows) and reads and writes three vectors
    bytes_it = n * e * (per_row + fill * (per_row + 1) / (1 if kind.startswith("g") else 2) + 6)
    flops_it = 2 * n * (per_row + fill * per_row + 5)
    if kind.startswith("g"):  # the Krylov basis, half a cycle on average: read once for the products, once after
        bytes_it += 2 * 15 * n * e
        flops_it += 4 * 15 * n
    it = _iterations(case)
    return {"bytes": it * bytes_it, "flops": it * flops_it}


def tolerance(case):
    """Products: four times the rounding measured against the stencil in 64
    bits (1e-16 and 7e-8 of the result, 8e-16 and 8e-7 in one entry).  Solves:
    four times the distance from x_true that the stopping test at 1e-8 leaves,
    which grows with the condition number: measured 4e-8 (37 x 31), up to 2.6e-6
    (128^2) and 1.2e-5 (600^2) in 2D, 1.4e-7 (20^3) to 2.7e-6 (100^3) in 3D, 2e-6
    for the batch's gradients; in one entry up to twenty times that."""
    if case["kind"] == "products":
        return {"rel": 5e-16, "max": 4e-15} if case["dtype"] == "f64" else {"rel": 3e-7, "max": 4e-6}
    if case["kind"] == "batch":
        seen = 2e-6
    else:
        s = max(case["nx"], case["ny"], case["nz"])
        seen = 2.6e-6 * (s / 128) ** 2 if case["nz"] == 1 else 2.7e-6 * s / 100
    return {"rel": 4 * seen, "max": 80 * seen}


# ----------------------------------------------------------------------------- exact answers
def _stencil_times(case, x, transpose):
    """A x (or A^T x) of the upwind convection-diffusion stencil, written out
    over the grid: diagonal 2 dim + h sum(beta), -1 - h beta_k upstream, -1 downstream."""
    nx, ny, nz, b = case["nx"], case["ny"], case["nz"], case["beta"]
    h = 1.0 / (nx + 1)
    beta = [b, b / 2] + ([b / 4] if nz > 1 else [])
    u = x.reshape(nz, ny, nx)
    y = (2 * len(beta) + h * sum(beta)) * u
    for k, bk in enumerate(beta):
        ax = 2 - k
        lo = [slice(None)] * 3
        hi = [slice(None)] * 3
        lo[ax], hi[ax] = slice(None, -1), slice(1, None)
        lo, hi = tuple(lo), tuple(hi)
        up, down = -1.0 - h * bk, -1.0
        if transpose:
            up, down = down, up
        y[hi] += up * u[lo]
        y[lo] += down * u[hi]
    return y.reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        J = _joined(_batch_systems(case, seed))
        n = len(J[0]) - 1
        x, lam = _truth(n, seed), _truth(n, seed, 1)
        rows = np.repeat(np.arange(n), np.diff(J[0]))
        return {"x": x, "grad_values": -lam[rows] * x[J[1]], "grad_b": lam}
    n = case["nx"] * case["ny"] * case["nz"]
    if kind == "products":
        x, b = _truth(n, seed), _truth(n, seed, 1)
        if case["dtype"] == "f32":
            x, b = x.astype(np.float32).astype(np.float64), b.astype(np.float32).astype(np.float64)
        y = _stencil_times(case, x, False)
        return {"y": y, "z": _stencil_times(case, y, True), "r": b - y}
    return _truth(n, seed)
