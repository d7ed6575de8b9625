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


@pytest.mark.parametrize("solver, use_graph", [("FCG", 1), ("FCG", 0), ("CGHS", 1), ("CGS", 1)])
@pytest.mark.parametrize("k", [1, 3])
def test_not_waited_for_again(solver, use_graph, k):
    """A call whose waits ended in vain is the last that waits: the next ones, and the rest of a solve, launch the
    sweeps one by one, with the same bits."""
    if solver == "CGS" and k > 1:
        pytest.skip("one column")
    L = bx.lib()
    patience, give_ups = L.bcmgx_internal_coarse_patience, L.bcmgx_internal_coarse_give_ups
    patience.argtypes = [bx.C.c_void_p, bx.C.c_longlong]
    give_ups.argtypes, give_ups.restype = [bx.C.c_void_p], bx.C.c_longlong
    ctx = bx.Context(0)
    n, row, col, val = bx.laplacian3d(7, 41, 40, 39)
    A = bx.CSR(ctx, n, n, row, col, val)
    p = bx.Params(solver=solver, preconditioner="BCMG", rtol=1e-8, check_every=2, sstep=2, use_graph=use_graph, dispnorm=0)
    P = bx.prec_setup(ctx, A, p)
    b = np.random.default_rng(3).normal(size=(n, k))
    solve = lambda: bx.solve(ctx, A, b, None, p, P)[0]
    x, u = solve(), P.apply(b)
    assert np.array_equal(solve(), x)  # replayed, where it is
    assert give_ups(ctx.h) == 0
    for call, result in ((solve, x), (lambda: P.apply(b), u)):
        before = give_ups(ctx.h)
        assert patience(ctx.h, -1) == 0
        for _ in range(3):
            assert np.array_equal(call(), result)
        assert give_ups(ctx.h) - before == 1
        assert patience(ctx.h, 500000) == 0
        for _ in range(2):
            assert np.array_equal(call(), result)
        assert give_ups(ctx.h) - before == 1
    P.finalize()
    A.close()
    ctx.close()


@pytest.mark.parametrize("widths, n_exchanges", [((64, 8), 1), ((64, 8, 3), 2), ((32, 8), 1), ((8, 64, 8), 2)])
def test_narrow_after_wide(widths, n_exchanges):
    """The exchange for a few columns does not depend on the widths before.  4096 rows run it to 8 columns (128 workgroups;
    16 as well with a HIP runtime whose occupancy query knows 160 KB of LDS a CU, so they are not asked for)."""
    L = bx.lib()
    patience, give_ups = L.bcmgx_internal_coarse_patience, L.bcmgx_internal_coarse_give_ups
    patience.argtypes = [bx.C.c_void_p, bx.C.c_longlong]
    give_ups.argtypes, give_ups.restype = [bx.C.c_void_p], bx.C.c_longlong
    ctx = bx.Context(0)
    n, row, col, val = bx.laplacian3d(27, 16, 16, 16)
    A = bx.CSR(ctx, n, n, row, col, val)
    P = bx.prec_setup(ctx, A, bx.Params(preconditioner="BCMG", max_levels=1, relaxnumber_coarse=20, dispnorm=0))
    for k in widths:
        f = np.random.default_rng(k).normal(size=(n, k))
        assert patience(ctx.h, 500000) == 0
        x = P.apply(f)
        assert patience(ctx.h, -1) == 0  # an exchange gives up at once, and says so
        assert np.array_equal(P.apply(f), x)
    assert give_ups(ctx.h) == n_exchanges
    P.finalize()
    A.close()
    ctx.close()
