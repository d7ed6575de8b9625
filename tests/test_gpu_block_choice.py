"""When the 16-row block form (csrc/blocked.hip) is made and how its use is chosen: a choice timed on one matrix serves
matrices of the same sharing of columns."""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu


def allocations(ctx, fail=-1):
    """device allocations of the context so far; the one after the next `fail` is to fail (-1: none)"""
    f = bx.lib().bcmgx_internal_fail_allocation
    f.argtypes = [bx.C.c_void_p, bx.C.c_longlong, bx.C.POINTER(bx.C.c_longlong)]
    count = bx.C.c_longlong()
    assert f(ctx.h, fail, bx.C.byref(count)) == 0
    return count.value


def test_choice_goes_by_the_sharing():
    """One grid in two numberings, the same rows and entries.  The timings take vectors of their own, so a solve that
    times allocates more than one whose choices are there."""
    ctx = bx.Context(0)
    dims = (43, 41, 39)
    n, row, col, val = bx.laplacian3d(27, *dims)
    S = sp.csr_matrix((val, col, row), shape=(n, n))
    order = np.random.default_rng(1).permutation(n)  # its tiles share other columns
    other = S[order][:, order].tocsr()
    other.sort_indices()
    p = bx.Params(solver="FCG", preconditioner="BCMG", precision="FP32", rtol=1e-6, dispnorm=0)
    counts = []
    for M in (S, S, other, other):
        A = bx.CSR.from_scipy(ctx, M)
        P = bx.prec_setup(ctx, A, p)
        before = allocations(ctx)
        assert bx.solve(ctx, A, np.ones((n, 16)), None, p, P)[1]["retv"] == 0
        counts.append(allocations(ctx) - before)
        P.finalize()
        A.close()
    ctx.close()
    assert counts[1] < counts[0] and counts[3] < counts[2]
