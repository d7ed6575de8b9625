"""The FP64 cycle's post sweep from A P (levels of 4 M entries and more) against the cycle without it, for one
and several columns, from zero and from a guess, and after A's values changed in place.

Tolerance: r_pre - (A P) e and f - A (x + P e) are the same sums grouped otherwise, each sweep rounding
some (row + 4) products of the values it combines; 100 of them cover a cycle's passes.
"""
import numpy as np
import pytest

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("points, dims", [(27, (57, 55, 51)), (7, (85, 85, 83)), (27, (53, 53, 53))])
@pytest.mark.parametrize("opt", [dict(), dict(prerelax_sweeps=2, postrelax_sweeps=2), dict(postrelax_sweeps=0), dict(cycle_type="W_CYCLE")],
                         ids=["default", "sweeps2", "no_post", "w"])
def test_cycle_as_without(ctx, points, dims, opt):
    n, row, col, val = bx.laplacian3d(points, *dims)
    A = bx.CSR(ctx, n, n, row, col, val)
    P = [bx.prec_setup(ctx, A, bx.Params(preconditioner="BCMG", dispnorm=0, post_galerkin=g, **opt)) for g in (1, 0)]
    rng = np.random.default_rng(n)
    for values in (val, val * 1.25):
        A.update_values(values)
        for k in (1, 3, 8):
            r, u = rng.normal(size=(n, k)), rng.normal(size=(n, k))
            for guess in (None, u):
                x, ref = (p.apply(r, guess) for p in P)
                assert np.abs(x - ref).max() <= 100 * (points + 4) * 2.0 ** -53 * np.abs(ref).max()
    for p in P:
        p.finalize()
    A.close()


def test_replayed_solves_see_new_values(ctx):
    n, row, col, val = bx.laplacian3d(27, 57, 55, 51)
    A = bx.CSR(ctx, n, n, row, col, val)
    p = bx.Params(preconditioner="BCMG", rtol=1e-10, dispnorm=0)
    P = bx.prec_setup(ctx, A, p)
    b = np.random.default_rng(2).normal(size=n)
    x = [bx.solve(ctx, A, b, None, p, P)[0] for _ in range(3)]
    assert np.array_equal(x[1], x[2])
    for scale in (2.0, 4.0, 0.5):  # a power of two scales every rounding with it
        A.update_values(val * scale)
        y, info = bx.solve(ctx, A, b, None, p, P)
        assert info["retv"] == 0
        r = b - scale * (A.to_scipy() / scale @ y)
        assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(b)
    P.finalize()
    A.close()
