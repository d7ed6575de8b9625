"""The coarsest level's l1-Jacobi sweeps in one launch (csrc/coarse.hip) against plain FP64 sweeps.

With max_levels = 1 the hierarchy is the matrix itself, so one preconditioner
application is relaxnumber_coarse sweeps x <- x + (f - A x) / M with M the row
sums of |A|.  Tolerance: a sweep rounds each row by at most (entries + 4) eps
of the values it combines and does not amplify (|I - A/M| <= 1 row-wise), so
s sweeps differ from any other order of the same sums by at most
s (maxrow + 4) eps max|x| (about 1e-12 at most here); FP32 rounds the result once.
"""
import numpy as np
import pytest

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu


def sweeps(S, f, x, s):
    M = np.asarray(abs(S).sum(axis=1)).ravel()
    for _ in range(s):
        x = (-(S @ x) + f) / M + x
    return x


# one workgroup (up to 4096 / lanes rows), its last size, the first exchanging one, a ragged last
# workgroup, many workgroups, past the resident limit (the launch-per-sweep path)
GRIDS = [(7, 1, 1, 1), (7, 4, 4, 4), (7, 8, 8, 8), (7, 9, 8, 8), (27, 8, 8, 4), (27, 5, 13, 4), (7, 13, 11, 17),
         (27, 16, 16, 16), (27, 19, 18, 17), (7, 32, 32, 32)]


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
@pytest.mark.parametrize("points,nx,ny,nz", GRIDS)
def test_coarsest_sweeps(ctx, points, nx, ny, nz, precision):
    n, row, col, val = bx.laplacian3d(points, nx, ny, nz)
    A = bx.CSR(ctx, n, n, row, col, val)
    S = A.to_scipy()
    rng = np.random.default_rng(n)
    for s in (2, 20, 64, 65):
        p = bx.Params(preconditioner="BCMG", precision=precision, max_levels=1, relaxnumber_coarse=s, dispnorm=0)
        P = bx.prec_setup(ctx, A, p)
        assert P.levels() == 1
        for rep in range(3):  # the exchange's tags rise from launch to launch
            f, u = rng.normal(size=n), rng.normal(size=n)
            if precision == "FP32":
                f, u = f.astype(np.float32).astype(float), u.astype(np.float32).astype(float)
            for guess in (None, u):
                x = P.apply(f, guess)
                ref = sweeps(S, f, np.zeros(n) if guess is None else guess, s)
                tol = s * (points + 4) * 2.3e-16 * np.abs(ref).max()
                if precision == "FP32":
                    tol += 6e-8 * np.abs(ref).max()
                assert np.abs(x - ref).max() <= tol, (s, rep, guess is None)
        P.finalize()
    A.close()


def test_coarsest_sweeps_unlisted_tiles(ctx):
    """Rows of up to 128 entries over scattered columns: tiles of 32 rows over the column list's
    limits (2048 entries, 1024 columns), beside listed ones."""
    import scipy.sparse as sp

    n, rng = 1500, np.random.default_rng(7)
    B = sp.random(n, n, density=0.03, random_state=rng, format="csr")
    T = sp.diags([np.ones(n - 1), np.ones(n - 1)], [-1, 1]).tocsr()
    S = abs(B + B.T).tolil()
    S[n // 2:] = 0
    S[:, n // 2:] = 0
    S = -(S.tocsr() + T)
    S.eliminate_zeros()
    S = (S + sp.diags(np.asarray(abs(S).sum(axis=1)).ravel() + 1.0)).tocsr()
    S.sort_indices()
    A = bx.CSR.from_scipy(ctx, S)
    maxrow = np.diff(S.indptr).max()
    P = bx.prec_setup(ctx, A, bx.Params(preconditioner="BCMG", max_levels=1, dispnorm=0))
    for _ in range(2):
        f = rng.normal(size=n)
        ref = sweeps(S, f, np.zeros(n), 20)
        assert np.abs(P.apply(f) - ref).max() <= 20 * (maxrow + 4) * 2.3e-16 * np.abs(ref).max()
    P.finalize()
    A.close()


@pytest.mark.parametrize("points,nx,ny,nz", [(7, 9, 8, 8), (27, 19, 18, 17)])
def test_waits_that_give_up(points, nx, ny, nz):
    """No waiting at all: the workgroup that finishes last computes the same bits, and the next
    launch exchanges again."""
    L = bx.lib()
    patience = L.bcmgx_internal_coarse_patience
    patience.argtypes = [bx.C.c_void_p, bx.C.c_longlong]
    ctx = bx.Context(0)
    n, row, col, val = bx.laplacian3d(points, nx, ny, nz)
    A = bx.CSR(ctx, n, n, row, col, val)
    P = bx.prec_setup(ctx, A, bx.Params(preconditioner="BCMG", max_levels=1, dispnorm=0))
    f = np.random.default_rng(1).normal(size=n)
    ref = P.apply(f)
    for _ in range(2):
        assert patience(ctx.h, -1) == 0
        assert np.array_equal(P.apply(f), ref)
        assert patience(ctx.h, 500000) == 0
        assert np.array_equal(P.apply(f), ref)
    P.finalize()
    A.close()
    ctx.close()
