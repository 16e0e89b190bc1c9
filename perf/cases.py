"""The work that users of the backend have it do, as cases that can be timed and checked.

A case is one of six kinds of call, each through the package's public entry points:

  solve    a Krylov solve on a kept matrix (Matrix.solve), as a program does for each right-hand side; with
           "update" new values go into the kept matrix first (Matrix.update_values), as in a time step
  oneshot  a Krylov solve from a host CSR (solve_csr): conversion, preconditioner set-up, solve
  spmv     y = A x on device arrays in one of the layouts
  step     the vector half of a hand-written Krylov loop on device vectors: q = A p with p.q, then the BLAS-1
  ilu0     ILU(0) factorisation and one triangular solve on device arrays with level-set schedules
  grad     one training gradient of the learned preconditioner (gnn_loss_grad)

Systems come from the package's generators. Solves whose rounding may travel through hundreds of iterations ask for a
tight residual (1e-12), so that the solution itself is determined; the ones of a few tens of iterations ask for 1e-8.
"""
import ctypes

import numpy as np
import torch

import alien_amd as aa

MATRIX = {"poisson": aa.GEN_POISSON7, "convdiff": aa.GEN_CONVDIFF7, "lognormal": aa.GEN_LOGNORMAL7}
SOLVER = {"cg": aa.CG, "bicgs": aa.BICGS}
PRECOND = {"diag": aa.PREC_DIAG, "cheb": aa.PREC_CHEB, "ilu0": aa.PREC_ILU0, "learned": aa.PREC_LEARNED}
MODE = {"reference": aa.MODE_REFERENCE, "fused": aa.MODE_FUSED, "graph": aa.MODE_GRAPH, "mixed": aa.MODE_MIXED}
LAYOUT = {"csr": aa.LAYOUT_CSR, "bellpack": aa.LAYOUT_BELLPACK, "rbdia": aa.LAYOUT_RBDIA}
LARGEST = 256**3  # rows of the largest listed system


def _solve(name, kind, dims, matrix, solver, precond, mode, tol, sigma=1.0, layout="rbdia", update=False, colours=False):
    nx, ny, nz = dims
    return {"name": name, "kind": kind, "nx": nx, "ny": ny, "nz": nz, "matrix": matrix, "sigma": sigma, "solver": solver,
            "precond": precond, "mode": mode, "layout": layout, "tol": tol, "update": update, "colours": colours}


def listed():
    return [
        # the smallest systems (the sizes of the learned preconditioner's training set and of the unit tests):
        # a solve is a string of short launches
        _solve("cg_jacobi_tiny", "solve", (14, 11, 9), "lognormal", "cg", "diag", "graph", 1e-12),
        # the plain method on a small grid: 32^3 Poisson, Chebyshev of degree 3, to 1e-8
        _solve("cg_cheb_poisson32", "solve", (32, 32, 32), "poisson", "cg", "cheb", "graph", 1e-8),
        # the drop-in algebra: one launch per call of Alien's templates, dots read back by the host, Alien's own CSR
        _solve("cg_reference_csr", "solve", (45, 38, 51), "poisson", "cg", "diag", "reference", 1e-12, layout="csr"),
        # a time step on a kept matrix: new values, then a mixed-precision solve
        _solve("step_mixed_jacobi64", "solve", (64, 64, 64), "lognormal", "cg", "diag", "mixed", 1e-12, update=True),
        # the largest: heterogeneous diffusion on 256^3 cells, learned preconditioner, FP32 inside FP64
        _solve("cg_learned_mixed256", "solve", (256, 256, 256), "lognormal", "cg", "learned", "mixed", 1e-12),
        # the nonsymmetric method: 128^3 upwind convection-diffusion, BiCGStab with the reference's own ILU(0)
        _solve("bicgs_ilu0_convdiff128", "solve", (128, 128, 128), "convdiff", "bicgs", "ilu0", "graph", 1e-8),
        # a matrix that is solved with once, from the host CSR: conversion, colouring, factorisation, CG
        _solve("oneshot_colour_ilu0_80", "oneshot", (80, 80, 80), "lognormal", "cg", "ilu0", "graph", 1e-12, colours=True),
        # the products themselves, on a user's own device arrays: Alien's CSR, and 2x2 blocks (two unknowns per cell)
        {"name": "spmv_csr_f64", "kind": "spmv", "layout": "csr", "fp32": False, "nx": 160, "ny": 160, "nz": 160},
        {"name": "spmv_bsr2_f64", "kind": "spmv", "layout": "bsr2", "fp32": False, "nx": 97, "ny": 93, "nz": 101},
        # one pass of a hand-written Krylov loop over an odd number of rows
        {"name": "step_vectors", "kind": "step", "nx": 101, "ny": 99, "nz": 103},
        # the triangular preconditioner through its own entry points
        {"name": "ilu0_factor_solve", "kind": "ilu0", "matrix": "convdiff", "nx": 64, "ny": 64, "nz": 64},
        # one training step's gradient: residual reduction after 16 preconditioned CG steps on a training-size system
        {"name": "train_grad", "kind": "grad", "nx": 16, "ny": 16, "nz": 16, "cg_steps": 16, "beta": 0.1},
    ]


def _edge(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _dims(rng, lo, hi):
    e = _edge(rng, lo, hi)
    return [max(lo, min(hi, e + rng.randint(-(e // 8) - 1, e // 8 + 1))) for _ in range(3)]


def draw(rng):
    """One more case of the same ranges: sizes over their logarithm, odd ones among them."""
    kind = rng.choice(["solve", "solve", "solve", "solve", "oneshot", "spmv", "spmv", "step", "ilu0", "grad"])
    if kind in ("solve", "oneshot"):
        form = rng.choice(["small", "small", "reference", "mixed", "learned", "ilu0"]) if kind == "solve" else "colours"
        if form == "small":
            matrix = rng.choice(["poisson", "lognormal"])
            precond = rng.choice(["diag", "cheb"]) if matrix == "poisson" else "diag"
            c = _solve("", kind, _dims(rng, 8, 72), matrix, "cg", precond, rng.choice(["graph", "fused"]), 1e-12,
                       sigma=round(rng.uniform(0.5, 1.0), 3))
        elif form == "reference":
            c = _solve("", kind, _dims(rng, 10, 64), "poisson", "cg", "diag", "reference", 1e-12,
                       layout=rng.choice(["csr", "bellpack"]))
        elif form == "mixed":
            c = _solve("", kind, _dims(rng, 16, 96), "lognormal", "cg", "diag", "mixed", 1e-12,
                       sigma=round(rng.uniform(0.5, 1.0), 3), update=rng.random() < 0.5)
        elif form == "learned":
            c = _solve("", kind, _dims(rng, 32, 160), "lognormal", "cg", "learned", "mixed", 1e-12,
                       sigma=round(rng.uniform(0.5, 1.0), 3), update=rng.random() < 0.5)
        elif form == "ilu0":
            c = _solve("", kind, _dims(rng, 16, 128), "convdiff", "bicgs", "ilu0", rng.choice(["graph", "fused", "reference"]), 1e-8)
        else:
            c = _solve("", kind, _dims(rng, 24, 96), "lognormal", "cg", "ilu0", rng.choice(["graph", "fused"]), 1e-12,
                       sigma=round(rng.uniform(0.5, 1.0), 3), colours=True)
        del c["name"]
        return c
    if kind == "spmv":
        nx, ny, nz = _dims(rng, 24, 176)
        layout = rng.choice(["csr", "csr", "bellpack", "rbdia", "bsr2"])
        if layout == "bsr2":
            nx, ny, nz = (max(12, int(e * 0.7)) for e in (nx, ny, nz))
        return {"kind": "spmv", "layout": layout, "fp32": rng.random() < 0.4, "nx": nx, "ny": ny, "nz": nz}
    if kind == "step":
        nx, ny, nz = _dims(rng, 16, 160)
        return {"kind": "step", "nx": nx, "ny": ny, "nz": nz}
    if kind == "ilu0":
        nx, ny, nz = _dims(rng, 12, 96)
        return {"kind": "ilu0", "matrix": rng.choice(["convdiff", "lognormal"]), "nx": nx, "ny": ny, "nz": nz}
    nx, ny, nz = _dims(rng, 8, 20)
    return {"kind": "grad", "nx": nx, "ny": ny, "nz": nz, "cg_steps": rng.choice([0, 8, 16, 40]), "beta": rng.choice([0.0, 0.1])}


_context = []


def _ctx():
    """The program's one context (a stream and the reductions' workspace)."""
    if not _context:
        _context.append(aa.Context())
    return _context[0]


class _State(dict):
    def __del__(self):
        if self.get("M") is not None:
            self["M"].close()


def _system(case, seed):
    """(row_offset, cols, vals) of the case's 7-point system."""
    matrix = case.get("matrix", "lognormal")
    par = [case.get("sigma", 1.0), 1.0, 1.0, 1.0] if matrix == "lognormal" else None
    return aa.gen_csr(MATRIX[matrix], case["nx"], case["ny"], case["nz"], params=par, seed=seed % (1 << 30))


def _product(ro, cols, vals, x):
    return np.add.reduceat(vals * x[cols], ro[:-1])


def _uniform(case, seed, n, stream=0):
    return np.random.default_rng([seed, stream]).random(n)


def _params(case):
    return {"solver": SOLVER[case["solver"]], "precond": PRECOND[case["precond"]], "layout": LAYOUT[case["layout"]],
            "mode": MODE[case["mode"]], "tol": case["tol"], "max_iter": 20000, "poll_every": 8,
            "ilu_schedule": 1 if case["colours"] else 0,
            "gnn_theta": aa.gnn_init(0) if case["precond"] == "learned" else None}


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _values(case, seed):
    """FP64 values of a new time step: the system's own, each face coefficient scaled by the step's factor."""
    return 1.0 + 0.5 * np.random.default_rng([seed, 9]).random()


def prepare(case, seed):
    ctx, s = _ctx(), _State(case=case)
    if case["kind"] in ("solve", "oneshot"):
        ro, cols, vals = _system(case, seed)
        if case["update"]:
            s["vals"] = vals * _values(case, seed)
        x = _uniform(case, seed, len(ro) - 1)
        s["b"] = _product(ro, cols, s.get("vals", vals), x)
        s["params"] = _params(case)
        if case["kind"] == "solve":
            s["M"] = aa.Matrix(ctx, ro, cols, vals)
        else:
            s["csr"] = (ro, cols, vals)
        return s
    if case["kind"] == "spmv":
        return _prepare_spmv(case, seed, s, ctx)
    if case["kind"] == "grad":
        ro, cols, vals = _system(case, seed)
        rng = np.random.default_rng([seed, 3])
        s["csr"] = (ro, cols, vals)
        s["theta"] = _theta(seed)
        s["probes"] = np.where(rng.random((len(ro) - 1, 4)) < 0.5, -1.0, 1.0).astype(np.float32)
        return s
    ro, cols, vals = _system(case, seed)
    n = len(ro) - 1
    s.update(n=n, ro=_dev(ro), cols=_dev(cols), vals=_dev(vals))
    new = lambda k: torch.empty(k, dtype=torch.float64, device="cuda")  # noqa: E731
    if case["kind"] == "step":
        for k, name in enumerate(("p", "x0", "r0", "d")):
            s[name] = _dev(_uniform(case, seed, n, k) - 0.5)
        s["alpha"] = float(_uniform(case, seed, 1, 8)[0])
        for name in ("q", "x", "r", "z"):
            s[name] = new(n)
        s["dots"] = new(3)
        return s
    dcol = aa.host_dcol(ro, cols)
    s["dcol"] = _dev(dcol)
    for part, upper in (("lower", False), ("upper", True)):
        ptr, rows = aa.group_by_level(*aa.host_levels(ro, cols, dcol, upper))
        s[part] = (len(ptr) - 1, np.ascontiguousarray(ptr, np.int32), _dev(rows.astype(np.int32)))
    s["y"] = _dev(_uniform(case, seed, n))
    s.update(lu=new(len(cols)), t=new(n), x=new(n))
    return s


def _theta(seed):
    """Parameters some way into a training run: the initial ones, moved."""
    th = aa.gnn_init(seed % 1000)
    return (th + 0.02 * np.random.default_rng([seed, 4]).standard_normal(len(th))).astype(np.float32)


def _spmv_inputs(case, seed):
    """(row_offset, cols, values, x): host arrays in the case's precision; BSR: 4 values per block."""
    if case["layout"] == "bsr2":
        ro, cols, vals = aa.gen_bsr2(case["nx"], case["ny"], case["nz"], params=[1.0, 0.3], seed=seed % (1 << 30))
        n = 2 * (len(ro) - 1)
    else:
        ro, cols, vals = _system(case, seed)
        n = len(ro) - 1
    kind = np.float32 if case["fp32"] else np.float64
    return ro, cols, vals.astype(kind), _uniform(case, seed, n).astype(kind)


def _prepare_spmv(case, seed, s, ctx):
    ro, cols, vals, x = _spmv_inputs(case, seed)
    suffix = "_f32" if case["fp32"] else "_f64"
    L, n = aa.lib(), len(ro) - 1
    s["x"], s["y"] = _dev(x), _dev(np.zeros_like(x))
    xy = [_ptr(s["x"]), _ptr(s["y"])]
    if case["layout"] in ("csr", "bsr2"):
        s["arrays"] = [_dev(ro), _dev(cols), _dev(vals)]
        s["call"] = (getattr(L, "alien_hip_spmv_" + case["layout"] + suffix), [ctx.h, n] + [_ptr(a) for a in s["arrays"]] + xy)
    elif case["layout"] == "bellpack":
        bro, bc, bv, _, _ = aa.bellpack_build(ro, cols, vals.astype(np.float64), 1024)
        s["arrays"] = [_dev(bro), _dev(bc), _dev(bv.astype(vals.dtype))]
        s["call"] = (getattr(L, "alien_hip_spmv_bellpack" + suffix), [ctx.h, n, 1024] + [_ptr(a) for a in s["arrays"]] + xy)
    else:
        bo, doff, dmask = aa.rbdia_build(ro, cols)
        d = [_dev(a) for a in (ro, cols, vals.astype(np.float64), bo, doff, dmask.view(np.int64))]
        bv = torch.empty(64 * int(bo[-1]), dtype=s["x"].dtype, device="cuda")
        torch.cuda.synchronize()
        aa.check(getattr(L, "alien_hip_rbdia_fill" + suffix)(ctx.h, n, *[_ptr(a) for a in d[:5]], _ptr(bv)))
        ctx.synchronize()
        s["arrays"] = [d[3], d[4], d[5], bv]
        s["call"] = (getattr(L, "alien_hip_spmv_rbdia" + suffix), [ctx.h, n] + [_ptr(a) for a in s["arrays"]] + xy)
    return s


def run(s):
    case, ctx = s["case"], _ctx()
    if case["kind"] == "solve":
        if case["update"]:
            s["M"].update_values(s["vals"])
        x, res = s["M"].solve(s["b"], **s["params"])
        return {"x": x, "converged": int(res["status"])}
    if case["kind"] == "oneshot":
        x, res = aa.solve_csr(ctx, *s["csr"], s["b"], **s["params"])
        return {"x": x, "converged": int(res["status"])}
    if case["kind"] == "spmv":
        f, args = s["call"]
        aa.check(f(*args))
        return s["y"]
    if case["kind"] == "grad":
        loss, parts, grad = aa.gnn_loss_grad(ctx, *s["csr"], s["theta"], s["probes"], beta=case["beta"], cg_steps=case["cg_steps"])
        return {"loss": float(loss), "parts": [float(v) for v in parts], "grad": grad}
    L, n, check = aa.lib(), s["n"], aa.check
    if case["kind"] == "step":
        dots = [ctypes.c_void_p(s["dots"].data_ptr() + 8 * k) for k in range(3)]
        check(L.alien_hip_copy_f64(ctx.h, n, _ptr(s["x0"]), _ptr(s["x"])))
        check(L.alien_hip_copy_f64(ctx.h, n, _ptr(s["r0"]), _ptr(s["r"])))
        check(L.alien_hip_spmv_dot_csr_f64(ctx.h, n, _ptr(s["ro"]), _ptr(s["cols"]), _ptr(s["vals"]), _ptr(s["p"]), _ptr(s["q"]), dots[0]))
        check(L.alien_hip_axpy_f64(ctx.h, n, s["alpha"], _ptr(s["p"]), _ptr(s["x"])))
        check(L.alien_hip_axpy_dot_f64(ctx.h, n, -s["alpha"], _ptr(s["q"]), _ptr(s["r"]), dots[1]))
        check(L.alien_hip_pointwise_mult_f64(ctx.h, n, _ptr(s["d"]), _ptr(s["r"]), _ptr(s["z"])))
        check(L.alien_hip_dot_f64(ctx.h, n, _ptr(s["r"]), _ptr(s["z"]), dots[2]))
        return {"q": s["q"], "x": s["x"], "r": s["r"], "z": s["z"], "dots": s["dots"]}
    (nl, lp, lr), (nu, up, ur) = s["lower"], s["upper"]
    A = [_ptr(s["ro"]), _ptr(s["cols"]), _ptr(s["dcol"])]
    check(L.alien_hip_copy_f64(ctx.h, len(s["cols"]), _ptr(s["vals"]), _ptr(s["lu"])))
    check(L.alien_hip_ilu0_factor_f64(ctx.h, n, *A, _ptr(s["lu"]), nl, aa._capi.iptr(lp), _ptr(lr)))
    check(L.alien_hip_ilu0_solve_f64(ctx.h, n, *A, _ptr(s["lu"]), nl, aa._capi.iptr(lp), _ptr(lr), nu, aa._capi.iptr(up),
                                     _ptr(ur), _ptr(s["y"]), _ptr(s["t"]), _ptr(s["x"])))
    return {"lu": s["lu"], "x": s["x"]}


def _iterations(case):
    """About how many iterations such a solve takes (the work of an iterative method is per iteration)."""
    edge = (case["nx"] * case["ny"] * case["nz"]) ** (1 / 3)
    if case["solver"] == "bicgs":
        return 8
    per_edge = {"diag": 3.4, "cheb": 1.2, "ilu0": 1.7, "learned": 1.9}[case["precond"]]
    if case["matrix"] == "lognormal":
        per_edge *= 1.0 + 0.8 * case["sigma"]
    return max(8, int(per_edge * edge * -np.log10(case["tol"]) / 8))


def work(case):
    """A solve: its host inputs and result once, and per iteration the operands of the products (values, no column
    indices: the grid gives them) and the vectors of the recurrence once each, in the precision they are held in."""
    n = case["nx"] * case["ny"] * case["nz"]
    nnz = aa.gen_nnz(aa.GEN_POISSON7, case["nx"], case["ny"], case["nz"])
    kind = case["kind"]
    if kind in ("solve", "oneshot"):
        word = 4 if case["mode"] == "mixed" else 8
        times = 2 if case["solver"] == "bicgs" else 1
        applies = {"diag": 0, "cheb": 3, "ilu0": 1, "learned": 1 + n / nnz}[case["precond"]]  # matrix-sized operands
        step = times * (1 + applies) * nnz * word + (12 if times == 2 else 8) * n * word
        flops = times * (1 + applies) * 2 * nnz + (20 if times == 2 else 10) * n
        setup = 16 * n + (8 * nnz if case["update"] else 0) + (12 * nnz if kind == "oneshot" else 0)
        return {"bytes": setup + _iterations(case) * step, "flops": _iterations(case) * flops}
    if kind == "spmv":
        word = 4 if case["fp32"] else 8
        if case["layout"] == "bsr2":
            return {"bytes": nnz * (4 * word + 4) + 4 * n + 4 * n * word, "flops": 8 * nnz}
        index = 0 if case["layout"] == "rbdia" else 4
        return {"bytes": nnz * (word + index) + 4 * n + 2 * n * word, "flops": 2 * nnz}
    if kind == "step":
        return {"bytes": 12 * nnz + 4 * n + 8 * 8 * n, "flops": 2 * nnz + 13 * n}
    if kind == "ilu0":
        return {"bytes": 8 * nnz + 3 * 4 * nnz + 3 * 8 * nnz + 40 * n, "flops": 5 * nnz}
    # forward and backward of the network (three layers of 64 x 32, features and heads beside them) and of the CG steps
    dense = 3 * (2 * 3 * 64 * 32) * n
    cg = case["cg_steps"] * 4 * 3 * 3 * 2 * nnz
    return {"bytes": 12 * nnz + 4 * 4 * n + 3 * 2 * 32 * 4 * n, "flops": dense + cg}


def exact(case, seed):
    if case["kind"] in ("solve", "oneshot"):
        return {"x": _uniform(case, seed, case["nx"] * case["ny"] * case["nz"]), "converged": None}
    if case["kind"] == "spmv":
        ro, cols, vals, x = _spmv_inputs(case, seed)
        vals, x = vals.astype(np.float64), x.astype(np.float64)
        if case["layout"] != "bsr2":
            return _product(ro, cols, vals, x)
        x2 = x.reshape(-1, 2)[cols]
        v = vals.reshape(-1, 2, 2)  # v[block, column, row]
        return np.add.reduceat(v[:, 0] * x2[:, :1] + v[:, 1] * x2[:, 1:], ro[:-1], axis=0).reshape(-1)
    if case["kind"] == "step":
        ro, cols, vals = _system(case, seed)
        n = len(ro) - 1
        p, x, r, d = (_uniform(case, seed, n, k) - 0.5 for k in range(4))
        a = float(_uniform(case, seed, 1, 8)[0])
        q = _product(ro, cols, vals, p)
        x, r = x + a * p, r - a * q
        z = d * r
        return {"q": q, "x": x, "r": r, "z": z, "dots": np.array([p @ q, r @ r, r @ z])}
    if case["kind"] == "ilu0":
        return _exact_ilu0(case, seed)
    return _exact_grad(case, seed)


def _exact_ilu0(case, seed):
    """ILU(0) of a 7-point matrix plane by plane of i + j + k: only the pivots change among the upper entries."""
    ro, cols, vals = _system(case, seed)
    n, lu = len(ro) - 1, vals.copy()
    row = np.repeat(np.arange(n), np.diff(ro))
    strides = (1, case["nx"], case["nx"] * case["ny"])
    at = {}
    for o in strides + tuple(-o for o in strides) + (0,):
        if o not in at:  # (a grid of one cell in a direction has no entries there)
            k = np.flatnonzero(cols - row == o)
            at[o] = np.full(n, -1)
            at[o][row[k]] = k
    i = np.arange(n)
    depth = i % case["nx"] + i // case["nx"] % case["ny"] + i // strides[2]
    order = np.argsort(depth, kind="stable")
    planes = np.split(order, np.cumsum(np.bincount(depth))[:-1])
    t = _uniform(case, seed, n).copy()
    for rows in planes:
        for o in strides[::-1]:
            k = at[-o][rows]
            have = rows[k >= 0]
            k = k[k >= 0]
            lu[k] /= lu[at[0][have - o]]
            lu[at[0][have]] -= lu[k] * lu[at[o][have - o]]
            t[have] -= lu[k] * t[have - o]
    x = t
    for rows in planes[::-1]:
        for o in strides:
            k = at[o][rows]
            have = rows[k >= 0]
            x[have] -= lu[k[k >= 0]] * x[have + o]
        x[rows] /= lu[at[0][rows]]
    return {"lu": lu, "x": x}


def _exact_grad(case, seed):
    """The network, the loss after the CG steps (or Kaporin's bound) and their gradient in 64 bits, by autograd."""
    ro, cols, vals = _system(case, seed)
    n = len(ro) - 1
    row = torch.from_numpy(np.repeat(np.arange(n), np.diff(ro)))
    col, v = torch.from_numpy(cols.astype(np.int64)), torch.from_numpy(vals)
    dinv = torch.zeros(n, dtype=torch.float64).index_add(0, row[row == col], v[row == col]).rsqrt()
    ahat = v * dinv[row] * dinv[col]
    off, low = row != col, row > col
    r, c, e = row[off], col[off], -ahat[off]
    sums = lambda k, w: torch.zeros(n, dtype=torch.float64).index_add(0, k, w)  # noqa: E731
    s = sums(r, e)
    most = torch.zeros(n, dtype=torch.float64).scatter_reduce(0, r, e, "amax")
    f = torch.stack([torch.ones_like(s), s, 1 - s, most, sums(r[c > r], e[c > r] ** 2), sums(r[c < r], e[c < r] ** 2)], 1)
    theta = torch.from_numpy(_theta(seed).astype(np.float64)).requires_grad_()
    w = torch.split(theta, [6 * 32, 32] + [64 * 32, 32] * 3 + [32, 1, 32, 32, 1])
    spread = lambda i, j, a, y: torch.zeros(n, y.shape[1], dtype=torch.float64).index_add(0, i, a[:, None] * y[j])  # noqa: E731
    h = torch.relu(f @ w[0].view(6, 32) + w[1])
    for k in (2, 4, 6):
        h = h + torch.relu(torch.cat([h, spread(r, c, e, h)], 1) @ w[k].view(64, 32) + w[k + 1])
    diag = torch.exp(h @ w[8] + w[9])
    li, lj = row[low], col[low]
    edge = -ahat[low] * (h[li] @ w[10] + h[lj] @ w[11] + w[12])
    G = lambda y: diag[:, None] * y + spread(li, lj, edge, y)  # noqa: E731
    Gt = lambda y: diag[:, None] * y + spread(lj, li, edge, y)  # noqa: E731
    A = lambda y: spread(row, col, ahat, y)  # noqa: E731
    rng = np.random.default_rng([seed, 3])
    V = torch.from_numpy(np.where(rng.random((n, 4)) < 0.5, -1.0, 1.0))
    if case["cg_steps"]:
        res, t = V, Gt(V)
        p, rho = G(t), (t * t).sum(0)
        for j in range(case["cg_steps"]):
            q = A(p)
            res = res - rho / (p * q).sum(0) * q
            if j + 1 < case["cg_steps"]:
                t = Gt(res)
                now = (t * t).sum(0)
                p, rho = G(t) + now / rho * p, now
        first = torch.log((res * res).sum(0) / (V * V).sum(0)).mean()
    else:  # tr(G^T A G): on a 7-point pattern two coupled rows of G share one column, the lower row's own
        trace = (diag**2).sum() + (edge**2).sum() + 2 * (ahat[low] * edge * diag[lj]).sum()
        first = torch.log(trace / n) - 2 * torch.log(diag).sum() / n
    probe = ((V - G(Gt(A(V)))) ** 2).mean()
    loss = first + case["beta"] * probe
    loss.backward()
    return {"loss": float(loss.detach()), "parts": [float(first.detach()), float(probe.detach())], "grad": theta.grad.numpy()}
