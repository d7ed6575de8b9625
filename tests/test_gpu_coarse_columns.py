"""The coarsest level's l1-Jacobi sweeps of k columns in one launch (csrc/coarse.hip) against plain FP64 sweeps.

As for one column (test_gpu_coarse.py): max_levels = 1 makes an application relaxnumber_coarse sweeps, and
s sweeps differ from any other order of the same sums by at most s (maxrow + 4) eps max|x|; FP32
rounds the result once.
"""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu


def lap(points, *dims):
    n, row, col, val = bx.laplacian3d(points, *dims)
    return sp.csr_matrix((val, col, row), shape=(n, n))


def heavy(n, band, seed):
    """`band` scattered entries in the first half of the rows (tiles over the kernel's places), tridiagonal after"""
    r = np.random.default_rng(seed)
    B = sp.random(n // 2, n // 2, density=band / (n // 2), random_state=r, format="csr")
    S = sp.block_diag([abs(B + B.T), sp.csr_matrix((n - n // 2, n - n // 2))]).tocsr()
    S = -(S + sp.diags([np.ones(n - 1), np.ones(n - 1)], [-1, 1])).tocsr()
    return (S + sp.diags(np.asarray(abs(S).sum(axis=1)).ravel() + 1.0)).tocsr()


# one row, a workgroup, a row more, ragged last workgroups, rows of up to 8, 27 and about 60 entries, tiles
# with more columns than places, too many workgroups for the exchange
MATRICES = {
    "one": lambda: lap(7, 1, 1, 1),
    "n32": lambda: lap(7, 8, 4, 1),
    "n33": lambda: lap(7, 33, 1, 1),
    "grid7": lambda: lap(7, 13, 11, 17),
    "grid27": lambda: lap(27, 16, 16, 16),
    "ragged27": lambda: lap(27, 19, 18, 17),
    "heavy": lambda: heavy(1500, 20, 1),
    "large": lambda: lap(7, 32, 32, 31),
}


def sweeps(S, f, x, s):
    M = np.asarray(abs(S).sum(axis=1))
    for _ in range(s):
        x = (-(S @ x) + f) / M + x
    return x


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
@pytest.mark.parametrize("name", sorted(MATRICES))
def test_columns(name, precision):
    L = bx.lib()
    patience = L.bcmgx_internal_coarse_patience
    patience.argtypes = [bx.C.c_void_p, bx.C.c_longlong]
    ctx = bx.Context(0)
    S = MATRICES[name]().tocsr()
    S.sort_indices()
    A = bx.CSR.from_scipy(ctx, S)
    n, widest = S.shape[0], np.diff(S.indptr).max()
    rng = np.random.default_rng(n)
    for s in (2, 20, 64):
        P = bx.prec_setup(ctx, A, bx.Params(preconditioner="BCMG", precision=precision, max_levels=1, relaxnumber_coarse=s, dispnorm=0))
        assert P.levels() == 1
        for k in (2, 8, 11, 64, 3):
            f, u = rng.normal(size=(n, k)), rng.normal(size=(n, k))
            if precision == "FP32":
                f, u = f.astype(np.float32).astype(float), u.astype(np.float32).astype(float)
            for guess in (None, u):
                ref = sweeps(S, f, np.zeros((n, k)) if guess is None else guess, s)
                tol = s * (widest + 4) * 2.3e-16 * np.abs(ref).max()
                if precision == "FP32":
                    tol += 6e-8 * np.abs(ref).max()
                x = P.apply(f, guess)
                assert np.abs(x - ref).max() <= tol, (s, k, guess is None)
                # no waiting at all: the workgroup that finishes last computes the same bits; then exchanged again
                assert patience(ctx.h, -1) == 0
                assert np.array_equal(P.apply(f, guess), x)
                assert patience(ctx.h, 500000) == 0
                assert np.array_equal(P.apply(f, guess), x)
        P.finalize()
    A.close()
    ctx.close()
