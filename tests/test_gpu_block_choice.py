"""When the 16-row block form (csrc/blocked.hip) is made and how its use is chosen: a choice timed on one matrix serves
matrices of the same sharing of columns, and an allocation that fails once refuses the form once."""
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


def test_a_failed_allocation_is_not_for_good(ctx):
    n, row, col, val = bx.laplacian3d(27, 9, 8, 7)
    k, order = 8, np.arange(n, dtype=np.int32)
    x, y, dots = np.ones((n, k), np.float32), np.zeros((n, k), np.float32), np.zeros((k, 3))
    p = lambda v: v.ctypes.data_as(bx.C.c_void_p)
    product = lambda A: bx.lib().bcmgx_internal_block_product(ctx.h, A.h, p(order), k, 1, p(x), None, None, p(y), p(dots))
    A = bx.CSR(ctx, n, n, row, col, val)
    before = allocations(ctx)
    assert product(A) == 0
    total = allocations(ctx) - before
    ref = y.copy()
    A.close()
    for fail in range(total):
        A = bx.CSR(ctx, n, n, row, col, val)
        allocations(ctx, fail)
        code = product(A)
        allocations(ctx)
        assert code != 0
        y[:] = 0
        assert product(A) == 0
        assert np.array_equal(y, ref)
        A.close()


def test_products_follow_new_values(ctx):
    """the form is kept with the matrix, its values (FP32 and FP64) change with the matrix's: twice and thrice the product, to
    the bit for a power of two, within the sums' rounding (28 eps of sum |a||x|) else"""
    n, row, col, val = bx.laplacian3d(27, 21, 19, 13)
    S = sp.csr_matrix((val, col, row), shape=(n, n))
    k, order = 16, np.arange(n, dtype=np.int32)
    r = np.random.default_rng(4)
    x, wr, dots = r.normal(size=(n, k)).astype(np.float32), r.normal(size=(2, n, k)), np.zeros((k, 3))
    p = lambda v: v.ctypes.data_as(bx.C.c_void_p)
    A = bx.CSR(ctx, n, n, row, col, val)
    for op, dtype, eps in ((1, np.float32, 2.0 ** -24), (5, np.float64, 2.0 ** -53)):
        first = None
        for scale in (1.0, 2.0, 3.0):
            A.update_values(val * scale)
            y = np.zeros((n, k), dtype)
            assert bx.lib().bcmgx_internal_block_product(ctx.h, A.h, p(order), k, op, p(x), p(wr), None, p(y), p(dots)) == 0
            first = y if first is None else first
            ref = scale * (S @ x.astype(np.float64))
            assert (abs(y - ref) <= 28 * eps * scale * (abs(S) @ abs(x.astype(np.float64)))).all()
            assert scale == 3.0 or np.array_equal(y, scale * first)
    A.close()
