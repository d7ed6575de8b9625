"""One device allocation fails, at any point of a setup: the call says so, or it makes do without, and whatever is
solved afterwards is right, also after the matrix's values change and in replayed iterations."""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu
ERR_ALLOC = -3


def fail(ctx, after):
    """the allocation after the next `after` fails (-1: none); the number of them so far"""
    f = bx.lib().bcmgx_internal_fail_allocation
    f.argtypes = [bx.C.c_void_p, bx.C.c_longlong, bx.C.POINTER(bx.C.c_longlong)]
    count = bx.C.c_longlong()
    assert f(ctx.h, after, bx.C.byref(count)) == 0
    return count.value


def solved(ctx, A, S, p, P, seed):
    """solution within the solver's bound of the true residual (1 % for its recurrence)"""
    b = np.random.default_rng(seed).normal(size=S.shape[0])
    x, info = bx.solve(ctx, A, b, np.zeros(len(b)), p, P)
    return info["retv"] == 0 and np.linalg.norm(b - S @ x) <= 1.01 * p.rtol * np.linalg.norm(b)


@pytest.mark.parametrize("precision, dims", [("FP64", (56, 55, 54)), ("FP32", (17, 16, 15))])
def test_setup(precision, dims):
    """An FP64 hierarchy keeps A P from 4 M entries on, 27 a row here; an FP32 one on every level."""
    ctx = bx.Context(0)
    n, row, col, val = bx.laplacian3d(27, *dims)
    S = sp.csr_matrix((val, col, row), shape=(n, n))
    A = bx.CSR(ctx, n, n, row, col, val)
    p = bx.Params(solver="FCG", preconditioner="BCMG", precision=precision, rtol=1e-7, prerelax_sweeps=1, postrelax_sweeps=1,
                  autotune=0, dispnorm=0)
    bx.prec_setup(ctx, A, p).finalize()
    before = fail(ctx, -1)
    bx.prec_setup(ctx, A, p).finalize()
    total = fail(ctx, -1) - before
    assert total > 50
    made_do = 0
    for after in range(total):
        fail(ctx, after)
        try:
            P = bx.prec_setup(ctx, A, p)
        except bx.BcmgxError as e:
            assert e.status == ERR_ALLOC
            continue
        finally:
            fail(ctx, -1)
        made_do += 1
        for scale in (1.0, 2.0):
            A.update_values(val * scale)
            for seed in (1, 2):  # launched, then replayed
                assert solved(ctx, A, scale * S, p, P, seed), (after, scale, seed)
        P.finalize()
        A.update_values(val)
    assert (made_do > 0) == (precision == "FP64")  # the products of an FP64 hierarchy are not needed
    A.close()
    ctx.close()


def test_new_values():
    """the same while the values change: an error leaves no product of the old values behind"""
    ctx = bx.Context(0)
    n, row, col, val = bx.laplacian3d(27, 17, 16, 15)
    S = sp.csr_matrix((val, col, row), shape=(n, n))
    A = bx.CSR(ctx, n, n, row, col, val)
    p = bx.Params(solver="FCG", preconditioner="BCMG", precision="FP32", rtol=1e-7, prerelax_sweeps=1, postrelax_sweeps=1,
                  autotune=0, dispnorm=0)
    P = bx.prec_setup(ctx, A, p)
    before = fail(ctx, -1)
    A.update_values(val)
    total = fail(ctx, -1) - before
    P.finalize()
    assert total > 0
    for after in range(total):
        P = bx.prec_setup(ctx, A, p)
        assert solved(ctx, A, S, p, P, 1) and solved(ctx, A, S, p, P, 2)
        fail(ctx, after)
        with pytest.raises(bx.BcmgxError):
            A.update_values(val * 2.0)
        fail(ctx, -1)
        assert solved(ctx, A, 2.0 * S, p, P, 3)  # the matrix has its new values
        A.update_values(val)
        assert solved(ctx, A, S, p, P, 4) and solved(ctx, A, S, p, P, 5)
        P.finalize()
    A.close()
    ctx.close()
