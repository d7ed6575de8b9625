"""Column counts that run with zero columns beside them (csrc/capi.cpp): every caller's column as solved and
applied alone, the caller's padding rows left as they were, results of the caller's columns only.

Tolerance: a column that stopped at ||r|| <= rtol ||b|| has ||x - A^-1 b|| <= cond(A) rtol ||A^-1 b||, so two
solves of it differ by at most twice that.  One cycle rounds some (row + 4) products of the values it
combines in each of its passes; 100 of them.
"""
import numpy as np
import pytest

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu
COND = {(7, (13, 11, 9)): 100.0, (27, (9, 8, 7)): 60.0}  # bounds from the operators' extreme eigenvalues


@pytest.mark.parametrize("k", [2, 4, 5, 7, 8, 9, 13, 31, 33, 61, 63, 64])
@pytest.mark.parametrize("solver, prec, precision", [("FCG", "BCMG", "FP32"), ("FCG", "BCMG", "FP64"), ("CGHS", "L1_JACOBI", "FP64"),
                                                     ("FCG", "AFSAI", "FP64")])
@pytest.mark.parametrize("points, dims", sorted(COND))
def test_as_alone(ctx, points, dims, solver, prec, precision, k):
    n, row, col, val = bx.laplacian3d(points, *dims)
    A = bx.CSR(ctx, n, n, row, col, val)
    rtol = 1e-9
    p = bx.Params(solver=solver, preconditioner=prec, precision=precision, rtol=rtol, itnlim=300, dispnorm=0)
    P = bx.prec_setup(ctx, A, p)
    r = np.random.default_rng(n + k)
    b, guess = r.normal(size=(n, k)), r.normal(size=(n, k))
    picks = sorted({0, k // 2, k - 1})
    for x0 in (None, guess):
        x, info = bx.solve(ctx, A, b, x0, p, P)
        assert info["retv"] == 0 and len(info["niter_cols"]) == k and info["niter"] == max(info["niter_cols"])
        for c in picks:
            one, _ = bx.solve(ctx, A, b[:, c], None if x0 is None else x0[:, c], p, P)
            assert np.linalg.norm(x[:, c] - one) <= 2.02 * COND[points, dims] * rtol * (1 if x0 is None else 100) * np.linalg.norm(one)
    ld = n + 5
    B, X = np.full((k, ld), 3.0), np.full((k, ld), 4.0)
    B[:, :n], X[:, :n] = b.T, 0.0
    dB, dX = bx.DeviceArray(ctx, (k * ld,)), bx.DeviceArray(ctx, (k * ld,))
    dB.upload(B.ravel())
    dX.upload(X.ravel())
    bx.solve_device(ctx, A, dB.ptr, dX.ptr, k, p, P, ld)
    got = dX.download().reshape(k, ld)
    assert np.all(got[:, n:] == 4.0)
    x, _ = bx.solve(ctx, A, b, None, p, P)
    assert np.linalg.norm(got[:, :n].T - x) <= 2.02 * COND[points, dims] * rtol * np.linalg.norm(x)
    eps = 2.0 ** -24 if precision == "FP32" else 2.0 ** -53
    for g in (None, guess):
        u = P.apply(b, g)
        for c in picks:
            one = P.apply(b[:, c], None if g is None else g[:, c])
            assert np.abs(u[:, c] - one.reshape(-1)).max() <= 100 * (points + 4) * 2 * eps * np.abs(one).max()
    P.finalize()
    A.close()


def test_a_limit_reached(ctx):
    n, row, col, val = bx.laplacian3d(7, 13, 11, 9)
    A = bx.CSR(ctx, n, n, row, col, val)
    b = np.random.default_rng(1).normal(size=(n, 5))
    for solver, prec in (("FCG", "BCMG"), ("CGHS", "BCMG")):
        p = bx.Params(solver=solver, preconditioner=prec, precision="FP32", rtol=1e-12, itnlim=2, dispnorm=0)
        P = bx.prec_setup(ctx, A, p)
        _, info = bx.solve(ctx, A, b, None, p, P)
        assert info["retv"] == -1 and len(info["niter_cols"]) == 5
        P.finalize()
    A.close()
