"""Waits of the one-launch coarsest sweeps (csrc/coarse.hip) that end before their values come: some workgroups
give up, at any sweep, while others go through, and the one that finishes last computes the sweeps.  The bits are
those of a launch in which nothing is waited for in vain."""
import numpy as np
import pytest

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
@pytest.mark.parametrize("k", [1, 2, 8, 11])
@pytest.mark.parametrize("points, dims", [(7, (33, 9, 4)), (27, (16, 16, 16)), (27, (19, 18, 17))])
def test_bounded_waits(points, dims, k, precision):
    patience = bx.lib().bcmgx_internal_coarse_patience
    patience.argtypes = [bx.C.c_void_p, bx.C.c_longlong]
    ctx = bx.Context(0)
    n, row, col, val = bx.laplacian3d(points, *dims)
    A = bx.CSR(ctx, n, n, row, col, val)
    P = bx.prec_setup(ctx, A, bx.Params(preconditioner="BCMG", precision=precision, max_levels=1, relaxnumber_coarse=20, dispnorm=0))
    f = np.random.default_rng(n).normal(size=(n, k))
    f = f[:, 0] if k == 1 else f
    x = P.apply(f)
    for ticks in (0, 50, 100, 200, 400, 1000) * 4:  # 100 MHz: a sweep takes some 200, so that waits end here and there
        assert patience(ctx.h, ticks) == 0
        assert np.array_equal(P.apply(f), x)
        assert patience(ctx.h, 500000) == 0
        assert np.array_equal(P.apply(f), x)  # nothing of it is left for the next launch
    P.finalize()
    A.close()
    ctx.close()
