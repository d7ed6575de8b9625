"""Solves and applications where memory is short: what a call can do without (zero columns beside its own, the
matrix's block form, the product A P of an FP64 hierarchy) is given up before the call is refused, and not asked for
again."""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu
MB = 1 << 20


def memory(ctx, limit):
    """allocations fail that bring the bytes in use over `limit` (0: none); the most in use since the last call"""
    f = bx.lib().bcmgx_internal_memory_limit
    f.argtypes = [bx.C.c_void_p, bx.C.c_longlong, bx.C.POINTER(bx.C.c_longlong)]
    peak = bx.C.c_longlong()
    assert f(ctx.h, limit, bx.C.byref(peak)) == 0
    return peak.value


def allocations(ctx):
    f = bx.lib().bcmgx_internal_fail_allocation
    f.argtypes = [bx.C.c_void_p, bx.C.c_longlong, bx.C.POINTER(bx.C.c_longlong)]
    count = bx.C.c_longlong()
    assert f(ctx.h, -1, bx.C.byref(count)) == 0
    return count.value


def problem(ctx, points, dims):
    n, row, col, val = bx.laplacian3d(points, *dims)
    return bx.CSR(ctx, n, n, row, col, val), sp.csr_matrix((val, col, row), shape=(n, n))


def check_solve(ctx, A, S, p, P, k, seed):
    """true residuals within the solver's bound (1 % for its recurrence)"""
    B = np.random.default_rng(seed).normal(size=(S.shape[0], k))
    x, info = bx.solve(ctx, A, B, None, p, P)
    assert info["retv"] == 0
    assert (np.linalg.norm(B - S @ x.reshape(B.shape), axis=0) <= 1.01 * p.rtol * np.linalg.norm(B, axis=0)).all()


# 21060 rows: 30 and 31 FP64 columns take 5 MB, 32 take 6; 7 FP32 columns of 74088 rows 2 MB, 8 take 3
@pytest.mark.parametrize("solver, precision, dims, k, as_it_is",
                         [("FCG", "FP64", (30, 27, 26), 31, 30), ("CGHS", "FP64", (30, 27, 26), 31, 30), ("FCG", "FP32", (42, 42, 42), 7, 4)])
def test_padded_columns(solver, precision, dims, k, as_it_is):
    """`as_it_is` columns need no others beside them: where they fit, k do, in proportion"""
    ctx = bx.Context(0)
    A, S = problem(ctx, 7, dims)
    p = bx.Params(solver=solver, preconditioner="BCMG", precision=precision, rtol=1e-7, dispnorm=0)
    P = bx.prec_setup(ctx, A, p)
    base = memory(ctx, 0)
    base = memory(ctx, 0)  # in use now
    check_solve(ctx, A, S, p, P, as_it_is, 1)
    need = memory(ctx, 0) - base
    count = allocations(ctx)
    check_solve(ctx, A, S, p, P, as_it_is, 2)
    again = allocations(ctx) - count
    P.finalize()
    P = bx.prec_setup(ctx, A, p)
    memory(ctx, 0)
    limit = base + need * k // as_it_is + 2 * MB  # 2 MB: sizes are rounded up, level by level
    memory(ctx, limit)
    check_solve(ctx, A, S, p, P, k, 3)
    count = allocations(ctx)
    for seed in (4, 5):
        check_solve(ctx, A, S, p, P, k, seed)
    assert allocations(ctx) - count == 2 * again  # what did not fit is not tried again
    u = P.apply(np.ones((S.shape[0], k)))
    assert np.isfinite(u).all()
    memory(ctx, 0)
    P.finalize()
    A.close()
    ctx.close()


@pytest.mark.parametrize("k", [8, 16])
def test_block_form(k):
    """a batch that runs from the matrix's block form where there is room for it, and fits without"""
    ctx = bx.Context(0)
    A, S = problem(ctx, 27, (43, 41, 39))
    p = bx.Params(solver="FCG", preconditioner="BCMG", precision="FP32", rtol=1e-7, autotune=0, dispnorm=0)
    P = bx.prec_setup(ctx, A, p)
    memory(ctx, 0)
    base = memory(ctx, 0)
    check_solve(ctx, A, S, p, P, k, 1)
    need = memory(ctx, 0) - base
    P.finalize()
    p = bx.Params(solver="FCG", preconditioner="BCMG", precision="FP32", rtol=1e-7, dispnorm=0)
    P = bx.prec_setup(ctx, A, p)
    memory(ctx, 0)
    memory(ctx, memory(ctx, 0) + need)
    for seed in (2, 3):
        check_solve(ctx, A, S, p, P, k, seed)
    memory(ctx, 0)
    P.finalize()
    A.close()
    ctx.close()


def large(ctx, **more):
    """an FP64 hierarchy that keeps A P of its finest level (from 4 M entries on), unless post_galerkin=0"""
    return bx.Params(solver="FCG", preconditioner="BCMG", precision="FP64", rtol=1e-7, prerelax_sweeps=1, postrelax_sweeps=1,
                     dispnorm=0, **more)


@pytest.mark.parametrize("solver, k, device", [("FCG", 1, False), ("FCG", 1, True), ("FCG", 2, False), ("FCG", 3, True), ("CGHS", 2, False),
                                               ("CGS", 1, False), ("apply", 1, False), ("apply", 2, False)])
def test_product_of_the_finest_level(solver, k, device):
    """what fits a hierarchy without the product fits one with it; the values of the matrix may change afterwards"""
    ctx = bx.Context(0)
    A, S = problem(ctx, 27, (56, 55, 54))
    n = S.shape[0]
    b = np.random.default_rng(1).normal(size=(n, k))
    dB, dX = bx.DeviceArray(ctx, (k * n,)), bx.DeviceArray(ctx, (k * n,))
    dB.upload(b.T.ravel())

    def call(p, P):
        if device:
            dX.upload(np.zeros(k * n))
        if solver == "apply":
            if not device:
                return P.apply(b)
            bx._check(bx.lib().bcmgx_prec_apply(P.h, dB.ptr, dX.ptr, k, n, bx.MEM_DEVICE), ctx)
        elif device:
            bx.solve_device(ctx, A, dB.ptr, dX.ptr, k, p, P, n)
        else:
            return bx.solve(ctx, A, b, None, p, P)[0]
        return dX.download().reshape(k, n).T

    method = {} if solver == "apply" else {"solver": solver, "sstep": 2} if solver == "CGS" else {"solver": solver}
    results, limit = [], 0
    for post in (0, 1):
        p = large(ctx, post_galerkin=post)
        for key, v in method.items():
            p.set(key, v)
        P = bx.prec_setup(ctx, A, p)
        memory(ctx, 0)
        if post:
            memory(ctx, limit + MB)
        results.append([call(p, P) for _ in range(3)])
        if post:
            memory(ctx, 0)
            A.update_values(A.to_scipy().data)
            results.append([call(p, P)])
        else:
            limit = memory(ctx, 0)
        P.finalize()
    for x in results[1] + results[2]:  # without the product: the same operations
        assert np.array_equal(x, results[0][0])
    A.close()
    ctx.close()


def test_setup():
    """a setup that finds no memory for the product's sake is made without"""
    ctx = bx.Context(0)
    A, S = problem(ctx, 27, (56, 55, 54))
    p = large(ctx, post_galerkin=0)
    memory(ctx, 0)
    P = bx.prec_setup(ctx, A, p)
    need = memory(ctx, 0)
    P.finalize()
    p = large(ctx)
    for limit in (need + MB, need + 20 * MB, need + 40 * MB, need + 60 * MB, need + 80 * MB):
        memory(ctx, limit)
        P = bx.prec_setup(ctx, A, p)
        memory(ctx, 0)
        check_solve(ctx, A, S, p, P, 1, 1)
        P.finalize()
    memory(ctx, need // 2)
    with pytest.raises(bx.BcmgxError):
        bx.prec_setup(ctx, A, p)
    memory(ctx, 0)
    A.close()
    ctx.close()
