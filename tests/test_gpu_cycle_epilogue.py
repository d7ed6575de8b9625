"""One column through the cycle, where the first sweep, the prolongation and the post-smoothing
sweep from A P ride on other kernels (csrc/spmv.hip, coarse.hip), against the same column among
three, where they are passes of their own.

Sizes: a few rows, one level's rows on both sides of the CSR-stream kernel's limits for R and A P
(65536 and 262144 rows).  Tolerance: the two round differently in at most some 70 products of a
cycle (8 levels of up to 6, 20 sweeps of the coarsest), each (row + 4) roundings; 100 of them.
"""
import numpy as np
import pytest

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu

GRIDS = [(7, 5, 4, 3), (27, 13, 9, 7), (7, 41, 41, 39), (27, 47, 45, 31), (7, 83, 81, 80), (27, 101, 53, 50)]
OPTIONS = [
    dict(),
    dict(prerelax_sweeps=2, postrelax_sweeps=2),
    dict(prerelax_sweeps=0, postrelax_sweeps=1),
    dict(prerelax_sweeps=1, postrelax_sweeps=0),
    dict(cycle_type="W_CYCLE"),
    dict(cycle_type="H_CYCLE"),
    dict(cycle_type="VARIABLE_V_CYCLE"),
    dict(post_galerkin=0),
    dict(relaxnumber_coarse=1),
    dict(relaxnumber_coarse=0),
]


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("opt", OPTIONS, ids=lambda o: "-".join(f"{k}{v}" for k, v in o.items()) or "default")
@pytest.mark.parametrize("precision, eps", [("FP64", 2.0 ** -53), ("FP32", 2.0 ** -24)])
def test_one_column_as_among_three(grid, opt, precision, eps):
    points, *dims = grid
    n, row, col, val = bx.laplacian3d(points, *dims)
    rng = np.random.default_rng(n)
    r = rng.normal(size=(n, 3))
    ctx = bx.Context(0)
    A = bx.CSR(ctx, n, n, row, col, val)
    P = bx.prec_setup(ctx, A, bx.Params(preconditioner="BCMG", precision=precision, dispnorm=0, **opt))
    for guess in (None, rng.normal(size=(n, 3))):
        ref = P.apply(r, guess)
        got = P.apply(np.ascontiguousarray(r[:, 1]), None if guess is None else np.ascontiguousarray(guess[:, 1]))
        tol = 100 * (points + 4) * 2 * eps * np.abs(ref[:, 1]).max()
        assert np.abs(got.reshape(-1) - ref[:, 1]).max() <= tol
    P.finalize()
    A.close()
    ctx.close()
