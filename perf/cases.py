"""The preconditioned-solve work that users of this library have it do, as timed cases.

A case names an operation ("op"), an operator ("matrix", its sizes) and the
options of the call.  The operators:

  conv3d  7-point upwind convection-diffusion on an nx x ny x nz grid, the
          library's main stencil; the velocities vary by cell.
  lap2d   5-point Laplacian on an nx x ny grid.
  mesh3d  ragged 3-D mesh: the points of a grid coupled to a random part of
          their 26 neighbours (about 5 to 25 entries a row, symmetric
          pattern, nonsymmetric values), as finite-element and CFD meshes
          in their natural order are.
  block3d 7-point stencil of dense bs x bs blocks (coupled unknowns a point).

Device-resident calls go through the C ABI's handles on device arrays;
drop-in calls through the reference's entry points on host arrays.
Right-hand sides are b = A x for a random x, so the solution of a solve is
known whatever the path to it.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import torch

import lace_amd as L

PREC = {"f64": L.LACE_F64, "f32": L.LACE_F32, "bf16": L.LACE_BF16, "f16": L.LACE_F16}
KIND = {"exact": L.TRSV_LEVEL, "jacobi": L.TRSV_JACOBI}

# Neighbour steps (dz, dy, dx) by ascending row distance.
FACES = [(-1, 0, 0), (0, -1, 0), (0, 0, -1), (0, 0, 1), (0, 1, 0), (1, 0, 0)]
CUBE = [(z, y, x) for z in (-1, 0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1) if (z, y, x) != (0, 0, 0)]


def listed():
    return [
        # one application of ILU factors on a small operator: the launches and the call
        {"name": "apply_small", "op": "apply", "matrix": "lap2d", "nx": 64, "ny": 64, "nz": 1, "prec": "f64",
         "kind": "jacobi", "trans": 0},
        # one product on a mesh of about the size of the reference's logged CFD matrix
        {"name": "spmv_mesh", "op": "spmv", "matrix": "mesh3d", "nx": 59, "ny": 61, "nz": 59, "prec": "f64"},
        # one application of ILU factors by exact triangular solves, the default, on a mesh
        {"name": "exact_mesh", "op": "apply", "matrix": "mesh3d", "nx": 43, "ny": 47, "nz": 45, "prec": "f64",
         "kind": "exact", "trans": 0},
        # a time step's new preconditioner and its first use, in 16-bit factor storage, on an odd grid
        {"name": "setup_grid_bf16", "op": "setup", "matrix": "conv3d", "nx": 100, "ny": 77, "nz": 53, "prec": "bf16",
         "kind": "jacobi", "trans": 0},
        # the same on a mesh in FP64
        {"name": "setup_mesh_f64", "op": "setup", "matrix": "mesh3d", "nx": 47, "ny": 45, "nz": 43, "prec": "f64",
         "kind": "jacobi", "trans": 0},
        # the default solver (FP64 FGMRES(50), exact solves) on a small system
        {"name": "solve_small", "op": "solve", "matrix": "lap2d", "nx": 64, "ny": 64, "nz": 1, "path": "exact"},
        # the mixed-precision solve at the benchmark's size
        {"name": "solve_mixed_grid", "op": "solve", "matrix": "conv3d", "nx": 128, "ny": 128, "nz": 128,
         "path": "mixed"},
        # the mixed-precision solve on a mesh
        {"name": "solve_mixed_mesh", "op": "solve", "matrix": "mesh3d", "nx": 53, "ny": 51, "nz": 55,
         "path": "mixed"},
        # FP64 solve and adjoint with the gradient of a loss by the operator's values
        {"name": "adjoint_grid", "op": "adjoint", "matrix": "conv3d", "nx": 64, "ny": 64, "nz": 64, "path": "f64"},
        # 32 right-hand sides: solve, adjoint and gradient
        {"name": "block_rhs", "op": "block", "matrix": "conv3d", "nx": 80, "ny": 72, "nz": 64, "path": "mixed"},
        # coupled unknowns: block ILU and FGMRES
        {"name": "solve_blocks", "op": "bsolve", "matrix": "block3d", "nx": 41, "ny": 47, "nz": 43, "bs": 5,
         "prec": "f32"},
        # the reference's own calls on host arrays: ParILU, then restarted Householder FGMRES
        {"name": "dropin", "op": "dropin", "matrix": "mesh3d", "nx": 24, "ny": 25, "nz": 23},
    ]


def _grid(rng, lo, hi):
    """Three unequal sides whose product is spread over [lo, hi] by its logarithm."""
    n = lo * (hi / lo) ** rng.random()
    a, b = rng.uniform(0.7, 1.4), rng.uniform(0.7, 1.4)
    s = n ** (1.0 / 3.0)
    return {"nx": max(3, int(s * a)), "ny": max(3, int(s * b)), "nz": max(3, int(s / (a * b)))}


def _plane(rng, lo, hi):
    n = lo * (hi / lo) ** rng.random()
    a = rng.uniform(0.6, 1.6)
    return {"nx": max(3, int(n ** 0.5 * a)), "ny": max(3, int(n ** 0.5 / a)), "nz": 1}


def draw(rng):
    op = rng.choice(["spmv", "apply", "setup", "solve", "solve", "adjoint", "block", "bsolve", "dropin"])
    if op in ("spmv", "apply", "setup"):
        m = rng.choice(["lap2d", "conv3d", "mesh3d"])
        if op == "spmv":
            g = _plane(rng, 1e6, 2e6) if m == "lap2d" else _grid(rng, *((8e5, 2e6) if m == "conv3d" else (1e5, 2.2e5)))
            return {"op": op, "matrix": m, **g, "prec": rng.choice(["f64", "f32"])}
        g = _plane(rng, 1e3, 4e5) if m == "lap2d" else _grid(rng, 1e3, 4e5 if m == "conv3d" else 1e5)
        c = {"op": op, "matrix": m, **g}
        kind = rng.choice(["exact", "jacobi"])
        prec = rng.choice(["f64", "f32"] if kind == "exact" else ["f64", "f32", "bf16", "f16"])
        return {**c, "prec": prec, "kind": kind, "trans": rng.choice([0, 0, 1])}
    if op == "solve":
        m = rng.choice(["lap2d", "conv3d", "mesh3d"])
        g = _plane(rng, 1e3, 8e3) if m == "lap2d" else _grid(rng, 2e3, 5e5 if m == "conv3d" else 1e5)
        return {"op": op, "matrix": m, **g, "path": rng.choice(["exact", "f64", "mixed", "mixed16", "mgs"])}
    if op == "adjoint":
        return {"op": op, "matrix": rng.choice(["conv3d", "mesh3d"]), **_grid(rng, 2e3, 1e5),
                "path": rng.choice(["f64", "mixed"])}
    if op == "block":
        return {"op": op, "matrix": rng.choice(["conv3d", "mesh3d"]), **_grid(rng, 4e3, 1e5),
                "path": rng.choice(["f32", "mixed"])}
    if op == "bsolve":
        return {"op": op, "matrix": "block3d", **_grid(rng, 1e3, 5e4), "bs": rng.choice([3, 4, 5]),
                "prec": rng.choice(["f64", "f32", "bf16"])}
    return {"op": op, "matrix": "mesh3d", **_grid(rng, 1e3, 2e4)}


# ------------------------------------------------------------------ operators
def _win(n, d):
    """Slices of the points that have a neighbour at step d, and of those neighbours."""
    return slice(max(0, -d), n - max(0, d)), slice(max(0, d), n - max(0, -d))


def _shift(T, step):
    """Every point's neighbour value at a step (dz, dy, dx); zero outside the grid."""
    out = torch.zeros_like(T) if isinstance(T, torch.Tensor) else np.zeros_like(T)
    a, b = zip(*(_win(T.shape[i], step[i]) for i in range(3)))
    out[a] = T[b]
    return out


def _coefs(case, seed):
    """({step: values}, {step: presence}, diagonal) of a scalar operator on its grid."""
    r = np.random.default_rng(seed)
    nz, ny, nx = case["nz"], case["ny"], case["nx"]
    shape = (nz, ny, nx)
    one = np.ones(shape, bool)
    if case["matrix"] == "lap2d":
        val = {s: -np.ones(shape) for s in FACES if s[0] == 0}
        diag = np.full(shape, 4.0)
        has = {s: _shift(one, s) for s in val}
    elif case["matrix"] == "conv3d":
        pe = {(-1, 0, 0): 0.5, (0, -1, 0): 1.0, (0, 0, -1): 2.0}
        val, diag = {}, np.full(shape, 6.0)
        for s in FACES:
            v = np.zeros(shape)
            if s in pe:
                v = pe[s] * r.uniform(0.75, 1.25, shape)
            val[s] = -1.0 - v
            diag += v
        has = {s: _shift(one, s) for s in val}
    else:
        # the mesh is the same for every seed, its values are not
        mesh = np.random.default_rng([nx, ny, nz])
        val, has, diag = {}, {}, np.full(shape, 0.05)
        for s in CUBE[:13]:
            t = (-s[0], -s[1], -s[2])
            keep = _shift(one, s) & (mesh.random(shape) < (0.9 if abs(s[0]) + abs(s[1]) + abs(s[2]) == 1 else 0.45))
            has[s], has[t] = keep, _shift(keep, t)
        for s in CUBE:
            val[s] = -r.uniform(0.5, 1.5, shape)
            diag += np.where(has[s], -val[s], 0.0)
        diag *= 1.2  # an implicit time step's share
    prec = case.get("prec", "f64")
    for s in val:
        val[s] = np.where(has[s], val[s], 0.0)
        if prec != "f64":
            val[s] = val[s].astype(np.float32).astype(np.float64)
    if prec != "f64":
        diag = diag.astype(np.float32).astype(np.float64)
    return val, has, diag


def _csr(case, val, has, diag):
    nx, ny = case["nx"], case["ny"]
    n = diag.size
    steps = sorted(list(val) + [(0, 0, 0)], key=lambda s: s[2] + nx * (s[1] + ny * s[0]))
    cols, vals, keep = (np.empty((n, len(steps)), t) for t in (np.int32, np.float64, bool))
    rows = np.arange(n, dtype=np.int32)
    for q, s in enumerate(steps):
        cols[:, q] = rows + (s[2] + nx * (s[1] + ny * s[0]))
        vals[:, q] = (diag if s == (0, 0, 0) else val[s]).reshape(-1)
        keep[:, q] = True if s == (0, 0, 0) else has[s].reshape(-1)
    row = np.zeros(n + 1, np.int32)
    np.cumsum(keep.sum(1), out=row[1:])
    return L.HostCSR(row, cols[keep], vals[keep])


def _times(val, diag, X):
    """A X for X of the grid's shape (and perhaps a last axis of columns)."""
    wide = X.ndim == 4
    Y = (diag[..., None] if wide else diag) * X
    for s, v in val.items():
        Y = Y + (v[..., None] if wide else v) * _shift(X, s)
    return Y


def _adjoint_coefs(val):
    return {(-s[0], -s[1], -s[2]): _shift(v, (-s[0], -s[1], -s[2])) for s, v in val.items()}


def _blocks(case, seed):
    return L.gen_bcsr7(case["nx"], case["ny"], case["nz"], case["bs"], seed=1 + seed % 1000003, sigma=0.1, shift=5.0)


# ------------------------------------------------------------------ prepare
def _dev(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a)).reshape(-1).to("cuda", dtype)


def _p(t):
    return C.c_void_p(t.data_ptr())


def _options(case):
    o = L.default_opts()
    o.rtol = 1e-8
    o.parilu_sweeps = _sweeps(case)
    path = case.get("path", "exact")
    if path in ("f64", "mgs"):
        o.trsv = L.TRSV_JACOBI
    if path == "mgs":
        o.krylov = 1
    if path in ("mixed", "mixed16"):
        o.search_max, o.restart_max, o.trsv, o.inner_iters = 10, 50, L.TRSV_JACOBI, 10
        o.prec_precond = L.LACE_F32 if path == "mixed" else L.LACE_BF16
    if case["op"] == "block":
        o.search_max, o.restart_max, o.trsv, o.prec_precond = 30, 20, L.TRSV_JACOBI, L.LACE_F32
        o.inner_iters = 10 if path == "mixed" else 0
    if case["op"] == "bsolve":
        o.search_max, o.restart_max, o.trsv, o.prec_precond = 40, 20, L.TRSV_JACOBI, PREC[case["prec"]]
    return o


def _sweeps(case):
    """Synchronous ParILU sweeps: 3 settle a stencil's factors, a mesh's longer rows take 8."""
    return 8 if case["matrix"] == "mesh3d" else 3


def _dropin(case, seed, val, has, diag, b):
    # quiet: the reference's progress lines are for its own post-processing
    L.check(L.lib().lace_set_option(b"matlab_log", 0), "matlab_log")
    par = L.GmresParam()
    par.search_max, par.restart_max, par.tol_type, par.rtol = 30, 20, 1, 1e-8
    par.reorth, par.user_csrtrsv_choice, par.precondition = 0, 0, 1
    return {"A": _csr(case, val, has, diag), "b": L.HostVec(b.reshape(-1)), "n": diag.size, "par": par}


def prepare(case, seed):
    op = case["op"]
    r = np.random.default_rng([seed, 1])
    st = {"case": case}
    if op == "bsolve":
        row, col, val = _blocks(case, seed)
        bs, nb = case["bs"], len(row) - 1
        x = r.standard_normal((nb, bs))
        b = np.add.reduceat(np.einsum("kij,kj->ki", val, x[col]), row[:-1], axis=0)
        st["S"] = L.Solver(L.HostBCSR(row, col, val, bs), _options(case))
        st["b"], st["x"] = _dev(b), torch.empty(nb * bs, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        return st
    val, has, diag = _coefs(case, seed)
    n = diag.size
    if op == "dropin":
        b = _times(val, diag, r.standard_normal(diag.shape))
        return {**st, **_dropin(case, seed, val, has, diag, b)}
    H = _csr(case, val, has, diag)
    st["n"] = n
    if op == "spmv":
        dt = torch.float64 if case["prec"] == "f64" else torch.float32
        st["A"] = L.DevCSRMatrix(H, PREC[case["prec"]])
        st["x"], st["y"] = _dev(r.standard_normal(n), dt), torch.zeros(n, dtype=dt, device="cuda")
    elif op in ("apply", "setup"):
        dt = torch.float64 if case["prec"] == "f64" else torch.float32
        st["P"] = L.ParILU(H, PREC[case["prec"]])
        st["r"], st["z"] = _dev(r.standard_normal(n), dt), torch.empty(n, dtype=dt, device="cuda")
        st["P"].sweeps(_sweeps(case))
    elif op in ("solve", "adjoint"):
        st["S"] = L.Solver(H, _options(case))
        st["b"] = _dev(_times(val, diag, r.standard_normal(diag.shape)))
        st["x"] = torch.empty_like(st["b"])
        if op == "adjoint":
            st["g"] = _dev(_times(_adjoint_coefs(val), diag, r.standard_normal(diag.shape)))
            st["lam"] = torch.empty_like(st["b"])
            st["dA"] = torch.empty(int(H.row[-1]), dtype=torch.float64, device="cuda")
    elif op == "block":
        st["S"] = L.Solver(H, _options(case))
        dv = {s: torch.as_tensor(v).cuda() for s, v in val.items()}
        dd = torch.as_tensor(diag).cuda()
        for key, vs in (("b", dv), ("g", _adjoint_coefs(dv))):
            X = torch.as_tensor(r.standard_normal((*diag.shape, L.NRHS))).cuda()
            st[key] = _times(vs, dd, X).reshape(-1).contiguous()
        st["x"], st["lam"] = torch.empty_like(st["b"]), torch.empty_like(st["b"])
        st["dA"] = torch.empty(int(H.row[-1]), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    return st


# ------------------------------------------------------------------ run
def _zero(t):
    """Zero initial guess, on the library's stream."""
    L.check(L.lib().lace_daxpby(t.numel(), 0.0, _p(t), 0.0, _p(t), _p(t)), "daxpby")


def _solve(st, b, x, trans=0):
    _zero(x)
    stats = L.SolverStats()
    L.check(L.lib().lace_solver_solve_trans(st["S"].h, _p(b), _p(x), trans, C.byref(stats)), "solve")
    if stats.converged != 1:
        raise L.LaceError("solve did not converge")
    return x


def _solve_block(st, b, x, trans):
    _zero(x)
    stats = L.BlockStats()
    L.check(L.lib().lace_solver_solve_block(st["S"].h, _p(b), _p(x), trans, C.byref(stats)), "solve_block")
    if stats.converged != 1:
        raise L.LaceError("block solve did not converge")
    return x


def run(st):
    case, lib = st["case"], L.lib()
    op = case["op"]
    if op == "spmv":
        L.check(lib.lace_csr_spmv(st["A"].h, 1.0, _p(st["x"]), 0.0, _p(st["y"])), "spmv")
        return st["y"]
    if op in ("apply", "setup"):
        P = st["P"]
        if op == "setup":
            P.reset()
            P.sweeps(_sweeps(case))
        L.check(lib.lace_parilu_apply(P.h, KIND[case["kind"]], 5, case["trans"], _p(st["r"]), _p(st["z"])), "apply")
        return st["z"]
    if op in ("solve", "bsolve"):
        st["S"].setup()
        return _solve(st, st["b"], st["x"])
    if op == "adjoint":
        st["S"].setup()
        x, lam = _solve(st, st["b"], st["x"]), _solve(st, st["g"], st["lam"], 1)
        L.check(lib.lace_solver_grad_values(st["S"].h, _p(lam), _p(x), _p(st["dA"])), "grad_values")
        return x, lam, st["dA"]
    if op == "block":
        st["S"].setup()
        x, lam = _solve_block(st, st["b"], st["x"], 0), _solve_block(st, st["g"], st["lam"], 1)
        L.check(lib.lace_solver_grad_values_block(st["S"].h, _p(lam), _p(x), _p(st["dA"])), "grad_values_block")
        return x, lam, st["dA"]
    # drop-in: factors from the ParILU call, U turned into CSR, then FGMRES
    A, Lm, Um, Ur, X = st["A"], L.DMatrix(), L.DMatrix(), L.DMatrix(), L.DMatrix()
    plog, glog = L.PrecondLog(), L.GmresLog()
    lib.data_PariLU_v0_3(A.ref(), C.byref(Lm), C.byref(Um), 1e-10, C.byref(plog))
    A.release_rowidx()
    L.check(lib.data_zmconvert(Um, C.byref(Ur), Um.storage_type, L.Magma_CSR), "zmconvert")
    Ur.storage_type, Ur.fill_mode = L.Magma_CSRU, L.MagmaUpper
    L.check(lib.data_zvinit(C.byref(X), st["n"], 1, 0.0, L.MagmaColMajor), "zvinit")
    L.check(lib.data_fgmres_householder_restart(A.ref(), st["b"].ref(), C.byref(X), C.byref(Lm), C.byref(Ur),
                                                C.byref(st["par"]), C.byref(glog)), "fgmres")
    L.check(lib.data_zmfree(C.byref(Ur)), "zmfree")
    return L.owned_to_numpy(X, kind="dense"), L.owned_to_numpy(Lm)[2], L.owned_to_numpy(Um)[2]


# ------------------------------------------------------------------ what a pass needs
def _size(case):
    n = case["nx"] * case["ny"] * case["nz"]
    if case["matrix"] == "block3d":
        return n * case["bs"], 7 * n * case["bs"] ** 2
    return n, {"lap2d": 5, "conv3d": 7, "mesh3d": 14} [case["matrix"]] * n


def work(case):
    """Values and pattern of the operator once, vectors once; the arithmetic of one product with what is read."""
    n, nnz = _size(case)
    op = case["op"]
    es = 8 if case.get("prec", "f64") == "f64" or op == "bsolve" else 4
    index = nnz // case["bs"] ** 2 if op == "bsolve" else nnz
    cols = {"adjoint": 4, "block": 4 * L.NRHS}.get(op, 2)
    out = nnz * 8 if op in ("adjoint", "block", "dropin") else 0
    return {"bytes": float(nnz * es + 4 * index + 4 * n + cols * n * es + out),
            "flops": 2.0 * nnz * max(1, cols // 2)}


def tolerance(case):
    op = case["op"]
    if op in ("spmv", "apply", "setup"):
        # sums of a few terms a row, in the type's rounding; 16-bit factors
        # may fall to the other neighbour where a 32-bit sum rounds differently
        return {"rel": {"f64": 4e-15, "f32": 2e-6}.get(case["prec"], 4e-3)}
    # solves stop at a relative residual of 1e-8: two correct ones differ by
    # that times the operator's conditioning
    return {"rel": 2e-5}


# ------------------------------------------------------------------ 64-bit values
def _ilu(val, diag, sweeps):
    """Synchronous ILU(0) sweeps: lower (unit) and upper coefficients by step, and U's diagonal."""
    low = [s for s in val if s < (0, 0, 0)]
    up = [s for s in val if s > (0, 0, 0)]
    lo, hi, ud = {s: val[s].copy() for s in low}, {s: val[s].copy() for s in up}, diag.copy()
    add = lambda a, b: (a[0] + b[0], a[1] + b[1], a[2] + b[2])  # noqa: E731
    for _ in range(sweeps):
        acc = {s: np.array(v) for s, v in val.items()}
        acc[(0, 0, 0)] = diag.copy()
        for a in low:
            for b in up:
                s = add(a, b)
                if s in acc:
                    acc[s] -= lo[a] * _shift(hi[b], a)
        nlo = {}
        for s in low:
            # products with k below the column: the closing one, l_ij u_jj, is not in the sum
            nlo[s] = np.where(val[s] != 0, acc[s] / np.where(_shift(ud, s) != 0, _shift(ud, s), 1.0), 0.0)
        nhi = {s: np.where(val[s] != 0, acc[s], 0.0) for s in up}
        lo, hi, ud = nlo, nhi, acc[(0, 0, 0)]
    return lo, hi, ud


def _tri(off, diag, r, sweeps):
    y = r / diag
    for _ in range(sweeps - 1 if sweeps else 10 ** 6):
        s = np.zeros_like(r)
        for step, v in off.items():
            s += v * _shift(y, step)
        new = (r - s) / diag
        if not sweeps and np.array_equal(new, y):
            break
        y = new
    return y


def exact(case, seed):
    op = case["op"]
    r = np.random.default_rng([seed, 1])
    if op == "bsolve":
        return r.standard_normal((case["nx"] * case["ny"] * case["nz"], case["bs"])).reshape(-1)
    if op == "solve":
        return r.standard_normal(_size(case)[0])
    val, has, diag = _coefs(case, seed)
    if op == "dropin":
        return r.standard_normal(diag.size), None, None
    if op == "spmv":
        x = r.standard_normal(diag.size).reshape(diag.shape)
        x = x if case["prec"] == "f64" else x.astype(np.float32).astype(np.float64)
        return _times(val, diag, x).reshape(-1)
    if op in ("apply", "setup"):
        x = r.standard_normal(diag.size).reshape(diag.shape)
        x = x if case["prec"] == "f64" else x.astype(np.float32).astype(np.float64)
        if case["matrix"] == "mesh3d" and case["kind"] == "exact" and diag.size > 120000:
            return None
        lo, hi, ud = _ilu(val, diag, _sweeps(case))
        one = np.ones_like(ud)
        k = 0 if case["kind"] == "exact" else 5
        if case["trans"]:
            y = _tri(_adjoint_coefs(hi), ud, x, k)
            z = _tri(_adjoint_coefs(lo), one, y, k)
        else:
            z = _tri(hi, ud, _tri(lo, one, x, k), k)
        return z.reshape(-1)
    cols = L.NRHS if op == "block" else 1
    x = r.standard_normal((*diag.shape, cols))
    lam = r.standard_normal((*diag.shape, cols))
    steps = sorted(list(val) + [(0, 0, 0)], key=lambda s: s[2] + case["nx"] * (s[1] + case["ny"] * s[0]))
    g, keep = np.empty((diag.size, len(steps))), np.empty((diag.size, len(steps)), bool)
    for q, s in enumerate(steps):
        g[:, q] = -(lam * _shift(x, s)).sum(-1).reshape(-1)
        keep[:, q] = True if s == (0, 0, 0) else has[s].reshape(-1)
    return x.reshape(-1), lam.reshape(-1), g[keep]
