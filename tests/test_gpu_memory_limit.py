"""Solves and applications where memory is short: what a call can do without (zero columns beside its own, the
matrix's block form) is given up before the call is refused, and not asked for again."""
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
    assert (np.linalg.norm(B - S @ x, axis=0) <= 1.01 * p.rtol * np.linalg.norm(B, axis=0)).all()


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
