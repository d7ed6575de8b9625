"""Reductions that finish in the reducing kernel (csrc/fcg.hip) at the edges of their counters: 1, 32, 33,
64 and 65 workgroups, to 1024 totals and past them, solves repeated on one workspace (the counters
are cleared by their last taker) and replayed from the captured iterations.

Tolerance: a column that stopped at ||r|| <= rtol ||b|| has ||x - A^-1 b|| <= cond(A) rtol ||A^-1 b||;
1 % on top covers the rounding of the recurrence.
"""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu
RTOL = 1e-9


# 512 elements a workgroup: n k / 512 rounded up
@pytest.mark.parametrize("dims, k", [((8, 8, 8), 1), ((32, 32, 16), 1), ((33, 32, 16), 1), ((16, 16, 16), 8), ((23, 16, 16), 9), ((32, 16, 16), 8), ((33, 16, 16), 8),
                                     ((65, 8, 8), 8), ((32, 32, 33), 1), ((17, 13, 11), 3)])
@pytest.mark.parametrize("solver, prec, graph", [("FCG", "BCMG", 1), ("FCG", "BCMG", 0), ("FCG", "NONE", 1), ("CGHS", "L1_JACOBI", 1),
                                                 ("CGHS", "BCMG", 0)])
def test_repeated_solves(ctx, dims, k, solver, prec, graph):
    n, row, col, val = bx.laplacian3d(7, *dims)
    lu = spla.splu(sp.csr_matrix((val, col, row), shape=(n, n)).tocsc())
    lam = [2 * (1 - np.cos(np.pi * np.array([1, d]) / (d + 1))) for d in dims]
    cond = sum(x[1] for x in lam) / sum(x[0] for x in lam)
    A = bx.CSR(ctx, n, n, row, col, val)
    p = bx.Params(solver=solver, preconditioner=prec, rtol=RTOL, itnlim=500, dispnorm=0, use_graph=graph)
    P = bx.prec_setup(ctx, A, p)
    r = np.random.default_rng(n + k)
    for _ in range(3):
        b = r.normal(size=(n, k))
        exact = lu.solve(b)
        x, info = bx.solve(ctx, A, b, None, p, P)
        assert info["retv"] == 0
        again, info2 = bx.solve(ctx, A, b, None, p, P)
        assert np.array_equal(x, again) and info2["niter"] == info["niter"]
        err = np.linalg.norm(x.reshape(n, k) - exact, axis=0)
        assert np.all(err <= 1.01 * cond * RTOL * np.linalg.norm(exact, axis=0))
    P.finalize()
    A.close()
