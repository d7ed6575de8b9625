"""What a user of this library has it do, as cases that can be timed and checked.

Kinds of case, each one pass through the public entry points:

* ``step``: a preconditioner set up on a resident matrix and k right-hand sides solved with it
  (time to solution of one system);
* ``solve``: right-hand sides solved on a hierarchy that was set up before (time steps, repeated loads);
* ``apply``: one application of a preconditioner, as inside a program's own Krylov method;
* ``spmm``: y = A x on k column-major columns;
* ``adjoint``: the differentiable solve, forward and backward, on CPU tensors as its interface has them.

Matrices are the 7- and 27-point operators on nx x ny x nz grids (x fastest): the constant Laplacians
(diagonal 6 or 26, neighbours -1, Dirichlet by omission), or 7-point diffusion with a conductivity per
face, ``lognormal`` (exp(2 g), g ~ N(0, 1)) or ``uniform`` on [0.5, 2], drawn from the seed.
"""
import itertools
import math

import numpy as np
import torch

import bootcmatchgx_amd as bx

DEV = "cuda:0"
_ctx = None


def _context():
    """One context for the process, as a program keeps it."""
    global _ctx
    if _ctx is None:
        _ctx = bx.Context(0)
    return _ctx


# ------------------------------------------------------------------ cases ---
def _case(name, kind, points, dims, coef="constant", k=1, **more):
    c = {"kind": kind, "points": points, "nx": dims[0], "ny": dims[1], "nz": dims[2], "coef": coef, "k": k,
         "precision": "FP64", "prec": "BCMG", "solver": "FCG", "sweeps": 1, "rtol": 1e-8}
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: the 10^3 regression problem with the default settings (4 + 4 sweeps, 1e-6)
        _case("lap7_10_step_default", "step", 7, (10, 10, 10), sweeps=4, rtol=1e-6),
        # a modest 3-D Poisson problem, all FP64
        _case("lap7_50_step_fp64", "step", 7, (50, 50, 50)),
        # a large system with one right-hand side, all FP64, by multigrid and by the approximate inverse
        _case("lap27_128_step_fp64", "step", 27, (128, 128, 128)),
        _case("lap27_128_step_afsai", "step", 27, (128, 128, 128), prec="AFSAI"),
        # strongly varying coefficients, mixed precision, one right-hand side, many iterations
        _case("diff7_160_step_fp32", "step", 7, (160, 160, 160), coef="lognormal", precision="FP32"),
        # the benchmark's workload: 32 right-hand sides at once on an FP32 hierarchy
        _case("lap27_128_k32_step_fp32", "step", 27, (128, 128, 128), k=32, precision="FP32"),
        # a few right-hand sides on a hierarchy that is kept
        _case("lap27_128_k8_solve_fp32", "solve", 27, (128, 128, 128), k=8, precision="FP32"),
        # plain CG with the one-level smoother, a ragged grid and an odd number of columns
        _case("lap7_ragged_k5_cg_l1", "solve", 7, (61, 50, 43), k=5, prec="L1_JACOBI", solver="CGHS"),
        # one V(1,1) cycle on a ragged grid, for a program with its own Krylov method
        _case("lap27_ragged_apply_fp64", "apply", 27, (101, 67, 53)),
        # the matrix products a program calls by themselves
        _case("lap27_128_spmv_fp64", "spmm", 27, (128, 128, 128)),
        _case("lap27_128_spmm32_fp64", "spmm", 27, (128, 128, 128), k=32),
        # gradients of a solve with respect to the right-hand side and the matrix values
        _case("diff7_128_adjoint_fp64", "adjoint", 7, (128, 128, 128), coef="uniform"),
    ]


def draw(rng):
    """A case of the same ranges: grids from 10^3 to 2.1 M rows (ragged, spread over their logarithm), 1 to 64 columns."""
    kind = rng.choice(["step", "step", "solve", "apply", "spmm", "adjoint"])
    n = math.exp(rng.uniform(math.log(1e3), math.log(2.1e6)))
    k = rng.choice([1, 1, 2, 3, 5, 8, 12, 16, 31, 32, 48, 64])
    prec = rng.choice(["BCMG", "BCMG", "BCMG", "BCMG", "AFSAI", "L1_JACOBI"])
    solver = rng.choice(["FCG", "FCG", "CGHS"])
    points = rng.choice([7, 27])
    coef = rng.choice(["constant", "uniform", "lognormal"]) if points == 7 else "constant"
    if kind in ("adjoint", "apply"):
        k = 1 if kind == "adjoint" else k
        solver = "FCG"
    if kind == "adjoint":
        points, prec = 7, "BCMG"
        coef = rng.choice(["constant", "uniform"])
    if prec != "BCMG":  # one-level methods: many iterations
        n = min(n, 1.5e5)
        coef = "constant" if coef == "lognormal" else coef
    if coef == "lognormal":
        n = min(n, 1e6)
        solver = "FCG"
    k = max(1, min(k, int(6.7e7 / n)))
    a, b = math.exp(rng.uniform(-0.4, 0.4)), math.exp(rng.uniform(-0.4, 0.4))
    nx = max(3, round((n * a) ** (1 / 3)))
    ny = max(3, round((n / nx * b) ** 0.5))
    nz = max(3, round(n / nx / ny))
    # an application's result is FP64 through and through; solves take either hierarchy
    precision = "FP32" if prec == "BCMG" and kind in ("step", "solve") and solver == "FCG" and rng.random() < 0.6 else "FP64"
    return _case(None, kind, points, (nx, ny, nz), coef, k, precision=precision, prec=prec, solver=solver,
                 sweeps=rng.choice([1, 1, 2, 4]), rtol=rng.choice([1e-6, 1e-8, 1e-8]))


# ----------------------------------------------------------------- inputs ---
def _gen(seed, what):
    return torch.Generator(device=DEV).manual_seed(1000003 * int(seed) + what)


def _stencil(case, seed):
    """(offsets, values): linear column offsets in column order, each with the operator's values on all rows
    as an (nz, ny, nx) tensor, 0 where the neighbour lies outside the grid."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    face = None
    if case["coef"] != "constant":
        g = _gen(seed, 1)

        def draw_faces(*shape):
            if case["coef"] == "lognormal":
                return torch.exp(2.0 * torch.randn(shape, generator=g, device=DEV, dtype=torch.float64))
            return 0.5 + 1.5 * torch.rand(shape, generator=g, device=DEV, dtype=torch.float64)

        face = {2: draw_faces(nz, ny, nx + 1), 1: draw_faces(nz, ny + 1, nx), 0: draw_faces(nz + 1, ny, nx)}
    offsets, values = [], []
    for d in itertools.product((-1, 0, 1), repeat=3):  # (dz, dy, dx): column order
        reach = sum(map(abs, d))
        if case["points"] == 7 and reach > 1:
            continue
        v = torch.zeros((nz, ny, nx), device=DEV, dtype=torch.float64)
        if reach == 0:
            v += 6.0 if case["points"] == 7 else 26.0
            if face:
                v = sum(f.narrow(a, 0, s) + f.narrow(a, 1, s) for a, (f, s) in
                        ((0, (face[0], nz)), (1, (face[1], ny)), (2, (face[2], nx))))
        else:
            inside = tuple(slice(max(0, -o), s - max(0, o)) for o, s in zip(d, (nz, ny, nx)))
            if face:
                axis = [a for a in range(3) if d[a]][0]
                f = face[axis].narrow(axis, 0 if d[axis] < 0 else 1, (nz, ny, nx)[axis])
                v[inside] = -f[inside]
            else:
                v[inside] = -1.0
        offsets.append((d[0] * ny + d[1]) * nx + d[2])
        values.append(v)
    return offsets, values


def _csr(offsets, values):
    """CSR arrays of the operator (int32 row pointers and columns, FP64 values) on the GPU."""
    vals = torch.stack([v.reshape(-1) for v in values], 1)
    n = vals.shape[0]
    there = vals != 0
    row = torch.zeros(n + 1, dtype=torch.int32, device=DEV)
    row[1:] = torch.cumsum(there.sum(1), 0)
    cols = torch.arange(n, device=DEV, dtype=torch.int32)[:, None] + torch.tensor(offsets, device=DEV, dtype=torch.int32)
    return row, cols[there], vals[there]


def _times(offsets, values, x):
    """A x in 64 bits for x of shape (k, n)."""
    n = x.shape[1]
    y = torch.zeros_like(x)
    for o, v in zip(offsets, values):
        lo, hi = max(0, -o), min(n, n - o)
        if lo < hi:
            y[:, lo:hi] += v.reshape(-1)[lo:hi] * x[:, lo + o:hi + o]
    return y


def _normal(case, seed, what):
    n = case["nx"] * case["ny"] * case["nz"]
    return torch.randn((case["k"], n), generator=_gen(seed, what), device=DEV, dtype=torch.float64)


def _rhs(case, seed, offsets, values):
    """(right-hand sides, their solution or None): N(0, 1) columns for the constant Laplacians; A times an
    N(0, 1) field where the coefficients vary."""
    if case["coef"] == "constant":
        return _normal(case, seed, 2), None
    x = _normal(case, seed, 3)
    return _times(offsets, values, x), x


def _params(case):
    return bx.Params(solver=case["solver"], preconditioner=case["prec"], precision=case["precision"], rtol=case["rtol"],
                     prerelax_sweeps=case["sweeps"], postrelax_sweeps=case["sweeps"], dispnorm=0)


def prepare(case, seed):
    ctx = _context()
    offsets, values = _stencil(case, seed)
    row, col, val = _csr(offsets, values)
    n, params = row.numel() - 1, _params(case)
    s = {"case": case, "ctx": ctx, "n": n, "params": params}
    if case["kind"] == "adjoint":
        from bootcmatchgx_amd import autograd

        x, lam = _normal(case, seed, 3), _normal(case, seed, 4)
        s["system"] = autograd.SPDSystem(n, row.cpu().numpy(), col.cpu().numpy(), val.cpu().numpy(), params, ctx=ctx)
        s["values"] = val.cpu().requires_grad_()
        s["b"] = _times(offsets, values, x)[0].cpu().requires_grad_()
        s["cotangent"] = _times(offsets, values, lam)[0].cpu()
        s["sparse_solve"] = autograd.sparse_solve
        return s
    torch.cuda.synchronize()  # the library has a stream of its own
    s["A"] = bx.CSR.from_device(ctx, n, n, col.numel(), row.data_ptr(), col.data_ptr(), val.data_ptr())
    if case["kind"] == "spmm":
        s["x"], s["y"] = _normal(case, seed, 2), torch.zeros((case["k"], n), device=DEV, dtype=torch.float64)
        s["A"].analyse()
    else:
        s["b"], _ = _rhs(case, seed, offsets, values)
        s["x"] = torch.zeros_like(s["b"])
        if case["kind"] != "step":
            s["prec"] = bx.prec_setup(ctx, s["A"], params)
    torch.cuda.synchronize()
    return s


def run(state):
    kind = state["case"]["kind"]
    if kind == "adjoint":
        x = state["sparse_solve"](state["values"], state["b"], state["system"])
        gv, gb = torch.autograd.grad(x, (state["values"], state["b"]), state["cotangent"])
        return {"x": x, "grad_values": gv, "grad_b": gb}
    ctx, A, x, k, n = state["ctx"], state["A"], state["x"], state["case"]["k"], state["n"]
    ptr = bx.C.c_void_p
    if kind == "spmm":
        A.spmm_device(ptr(x.data_ptr()), ptr(state["y"].data_ptr()), k, n)
        return state["y"]
    b = state["b"]
    x.zero_()  # the zero guess
    torch.cuda.current_stream().synchronize()  # the library has a stream of its own
    if kind == "apply":
        bx._check(bx.lib().bcmgx_prec_apply(state["prec"].h, ptr(b.data_ptr()), ptr(x.data_ptr()), k, n, bx.MEM_DEVICE), ctx)
        return x
    prec = state["prec"] if kind == "solve" else bx.prec_setup(ctx, A, state["params"])
    bx.solve_device(ctx, A, ptr(b.data_ptr()), ptr(x.data_ptr()), k, state["params"], prec)
    if kind == "step":
        prec.finalize()
    return x


# ------------------------------------------------------------------- work ---
def _nnz(case):
    n = (case["nx"], case["ny"], case["nz"])
    if case["points"] == 27:
        return math.prod(3 * s - 2 for s in n)
    return math.prod(n) + 2 * sum(math.prod(n) // s * (s - 1) for s in n)


def _iterations(case):
    """Krylov iterations that these settings take, about: what the mathematics of the method needs."""
    side = (case["nx"] * case["ny"] * case["nz"]) ** (1 / 3)
    digits = -math.log10(case["rtol"]) / 8
    if case["prec"] == "BCMG":
        return max(3, digits * side ** 0.5 * (12 if case["coef"] == "lognormal" else 3.2) / case["sweeps"] ** 0.4)
    return max(3, digits * side * (0.7 if case["prec"] == "AFSAI" else 1.0))


def work(case):
    n, nnz, k = case["nx"] * case["ny"] * case["nz"], _nnz(case), case["k"]
    matrix, column = 12 * nnz + 4 * (n + 1), 8 * n
    if case["kind"] == "spmm":
        return {"bytes": matrix + 2 * k * column, "flops": 2 * nnz * k}
    if case["kind"] == "apply":  # the matrix once for the residual, once for the smoother after the correction
        return {"bytes": 2 * matrix + 2 * k * column, "flops": 4 * nnz * k}
    # an iteration: the matrix once for the product and once for the cycle's residual (in FP32 there, if so set);
    # p, w, z, A z and r read, and p, w, r and x written
    one = matrix + (matrix - 4 * nnz if case["precision"] == "FP32" else matrix) + 9 * k * column
    flops = 4 * nnz * k + 14 * n * k
    its = _iterations(case) * (2 if case["kind"] == "adjoint" else 1)
    setup = 2 * matrix if case["kind"] == "step" else 0
    if case["kind"] == "adjoint":
        setup = 2 * 8 * nnz  # the values in, their gradient out
    return {"bytes": its * one + setup, "flops": its * flops}


# ------------------------------------------------------------------ exact ---
def _sine_solve(case, b):
    """A^{-1} b of the constant Laplacians: the sine vectors of each direction diagonalise them."""
    nx, ny, nz, k = case["nx"], case["ny"], case["nz"], b.shape[0]

    def sines(s):
        j = torch.arange(1, s + 1, device=DEV, dtype=torch.float64)
        return math.sqrt(2.0 / (s + 1)) * torch.sin(math.pi / (s + 1) * j[:, None] * j), torch.cos(math.pi / (s + 1) * j)

    (sx, cx), (sy, cy), (sz, cz) = sines(nx), sines(ny), sines(nz)
    cx, cy, cz = cx[None, None, :], cy[None, :, None], cz[:, None, None]
    if case["points"] == 7:
        lam = 6 - 2 * (cx + cy + cz)
    else:
        lam = 27 - (1 + 2 * cx) * (1 + 2 * cy) * (1 + 2 * cz)

    def transform(u):
        u = (u.reshape(-1, nx) @ sx).reshape(k, nz, ny, nx)
        u = (u.transpose(2, 3).reshape(-1, ny) @ sy).reshape(k, nz, nx, ny).transpose(2, 3)
        return (u.transpose(1, 3).reshape(-1, nz) @ sz).reshape(k, nx, ny, nz).transpose(1, 3)

    return transform(transform(b.reshape(k, nz, ny, nx)) / lam).reshape(k, -1)


def exact(case, seed):
    if case["kind"] == "apply":
        return None  # what one cycle gives is defined by the method, not by A
    offsets, values = _stencil(case, seed)
    if case["kind"] == "spmm":
        return _times(offsets, values, _normal(case, seed, 2))
    if case["kind"] == "adjoint":
        x, lam = _normal(case, seed, 3)[0], _normal(case, seed, 4)[0]
        row, col, _ = _csr(offsets, values)
        i = torch.repeat_interleave(torch.arange(x.numel(), device=DEV), (row[1:] - row[:-1]).long())
        return {"x": x, "grad_values": -lam[i] * x[col.long()], "grad_b": lam}
    b, x = _rhs(case, seed, offsets, values)
    return x if x is not None else _sine_solve(case, b)
