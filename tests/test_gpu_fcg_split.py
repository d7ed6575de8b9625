"""The streaming FCG/CG kernels' split of n x k elements (csrc/fcg.hip) at its edges: any number of
columns per block, sizes around one block's 512 elements and many blocks.

Tolerance: a column that stopped at ||r|| <= rtol ||b|| has ||x - A^-1 b|| <= cond(A) rtol ||A^-1 b||;
1 % on top covers the rounding of the recurrence (cond eps64 is below 1e-13 on these grids).
"""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu
RTOL = 1e-9


@pytest.mark.parametrize("dims", [(3, 1, 1), (5, 4, 3), (17, 5, 3), (8, 8, 8), (19, 9, 3), (37, 29, 11)])
@pytest.mark.parametrize("k", [1, 2, 3, 5, 7, 16, 31, 33, 63, 64])
@pytest.mark.parametrize("solver, prec", [("FCG", "FP64"), ("FCG", "FP32"), ("CGHS", "FP64")])
def test_columns_against_direct(dims, k, solver, prec):
    n, row, col, val = bx.laplacian3d(7, *dims)
    A = sp.csr_matrix((val, col, row), shape=(n, n)).tocsc()
    b = np.random.default_rng(n * 100 + k).normal(size=(n, k))
    b[:, k // 2] = 0.0 if k > 1 else b[:, 0]  # a column that stops at once
    exact = spla.splu(A).solve(b)
    lam = [2 * (1 - np.cos(np.pi * np.array([1, d]) / (d + 1))) for d in dims]  # 7-point: sum over axes
    cond = sum(x[1] for x in lam) / sum(x[0] for x in lam)
    ctx = bx.Context(0)
    dA = bx.CSR(ctx, n, n, row, col, val)
    p = bx.Params(solver=solver, preconditioner="L1_JACOBI" if solver == "CGHS" else "BCMG", precision=prec, rtol=RTOL,
                  itnlim=500, dispnorm=0)
    P = bx.prec_setup(ctx, dA, p)
    x, info = bx.solve(ctx, dA, b, None, p, P)
    assert info["retv"] == 0
    err = np.linalg.norm(x.reshape(n, k) - exact, axis=0)
    assert np.all(err <= 1.01 * cond * RTOL * np.linalg.norm(exact, axis=0))
    P.finalize()
    dA.close()
    ctx.close()
