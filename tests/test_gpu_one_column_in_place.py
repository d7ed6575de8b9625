"""Applications and solves of one device column where it lies, against the staged ones of host arrays: equal
bits, r and b untouched, the guess taken from u, overlapping columns staged."""
import numpy as np
import pytest

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu
PARAMS = [dict(preconditioner="BCMG"), dict(preconditioner="BCMG", precision="FP32"), dict(preconditioner="BCMG", max_levels=1),
          dict(preconditioner="BCMG", postrelax_sweeps=0), dict(preconditioner="AFSAI"), dict(preconditioner="L1_JACOBI", l1jacsweeps=3),
          dict(preconditioner="L1_JACOBI", l1jacsweeps=4), dict(preconditioner="NONE"),
          dict(preconditioner="BCMG", max_hrc=2, conv_ratio=0.0, bootstrap_type="ADDITIVE"),
          dict(preconditioner="BCMG", max_hrc=2, conv_ratio=0.0, bootstrap_type="SYMMETRIZED_MULTIPLICATIVE")]


def device(ctx, a):
    d = bx.DeviceArray(ctx, (a.size,))
    d.upload(a)
    return d


@pytest.mark.parametrize("kw", PARAMS, ids=lambda k: "-".join(str(v) for v in k.values()))
@pytest.mark.parametrize("dims", [(3, 2, 1), (23, 19, 17)])
def test_apply_and_solve(ctx, dims, kw):
    n, row, col, val = bx.laplacian3d(7, *dims)
    A = bx.CSR(ctx, n, n, row, col, val)
    p = bx.Params(rtol=1e-8, itnlim=200, dispnorm=0, **kw)
    P = bx.prec_setup(ctx, A, p)
    rng = np.random.default_rng(n)
    r, u = rng.normal(size=n), rng.normal(size=n)
    dr, du = device(ctx, r), device(ctx, u)
    want = P.apply(r, u).reshape(-1)
    bx._check(bx.lib().bcmgx_prec_apply(P.h, dr.ptr, du.ptr, 1, n, bx.MEM_DEVICE), ctx)
    assert np.array_equal(du.download(), want) and np.array_equal(dr.download(), r)
    same = device(ctx, r)
    bx._check(bx.lib().bcmgx_prec_apply(P.h, same.ptr, same.ptr, 1, n, bx.MEM_DEVICE), ctx)
    assert np.array_equal(same.download(), P.apply(r, r).reshape(-1))
    for solver in ("FCG", "CGHS"):
        q = bx.Params(solver=solver, rtol=1e-8, itnlim=200, dispnorm=0, **kw)
        want, info = bx.solve(ctx, A, r, u, q, P)
        dx = device(ctx, u)
        got = bx.solve_device(ctx, A, dr.ptr, dx.ptr, 1, q, P)
        assert got["niter"] == info["niter"] and np.array_equal(dx.download(), want) and np.array_equal(dr.download(), r)
    P.finalize()
    A.close()
