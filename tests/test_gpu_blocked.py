"""k-column products from the 16-row block form (csrc/blocked.hip) against FP64 sums.

Tolerance: an FP32 sum of len products carries at most (len + 1) eps32 of sum |a||x|; the epilogue
adds two roundings of |b| and the result (three more with the division of the Jacobi sweep); FP64
sums the same with eps64, a dot product n + 1 roundings of sum |r||x|.
"""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu
E32, E64 = 2.0 ** -24, 2.0 ** -53


def lap(points, *dims):
    n, row, col, val = bx.laplacian3d(points, *dims)
    return sp.csr_matrix((val, col, row), shape=(n, n))


def scattered(n, per_row, seed):
    """per_row entries in random columns (tiles of up to 16 per_row distinct columns), some rows empty"""
    r = np.random.default_rng(seed)
    rows = [np.sort(r.choice(n, size=min(n, per_row if i % 7 else 0), replace=False)) for i in range(n)]
    ptr = np.concatenate([[0], np.cumsum([len(x) for x in rows])])
    return sp.csr_matrix((r.normal(size=ptr[-1]), np.concatenate(rows), ptr), shape=(n, n))


# one row; a tile but one, a tile, a tile and a row; ragged grids; tiles with the most entries (512)
# and columns; more than 16 groups of columns by one; tiles without entries
MATRICES = {
    "one": lambda: sp.csr_matrix(np.array([[2.5]])),
    "n15": lambda: lap(27, 5, 3, 1),
    "n16": lambda: lap(27, 4, 2, 2),
    "n17": lambda: lap(7, 17, 1, 1),
    "grid27": lambda: lap(27, 21, 19, 13),
    "grid7": lambda: lap(7, 40, 13, 7),
    "dense32": lambda: scattered(900, 32, 1),
    "dense4": lambda: scattered(333, 4, 2),
    "full17": lambda: sp.csr_matrix(np.random.default_rng(3).normal(size=(17, 17))),
    "wide65": lambda: sp.csr_matrix((np.ones(64 * 16 // 16 + 1), (np.arange(65) % 16, np.arange(65))), shape=(65, 65)),
    "empty_tiles": lambda: sp.csr_matrix((np.ones(3), ([0, 100, 101], [5, 7, 101])), shape=(130, 130)),
}


@pytest.mark.parametrize("k", [8, 16, 32, 64])
@pytest.mark.parametrize("name", sorted(MATRICES))
def test_block_products(ctx, name, k):
    S = MATRICES[name]().tocsr()
    S.sort_indices()
    n = S.shape[0]
    f = bx.lib().bcmgx_internal_block_product
    r = np.random.default_rng(k + n)
    for order in (np.arange(n), r.permutation(n)):
        order = order.astype(np.int32)
        A = bx.CSR.from_scipy(ctx, S)

        def product(op, x, b, D):
            y, dots = np.zeros((n, k), np.float64 if op == 5 else np.float32), np.zeros((k, 3))
            p = lambda v: None if v is None else v.ctypes.data_as(bx.C.c_void_p)
            assert f(ctx.h, A.h, p(order), k, op, p(x), p(b), p(D), p(y), p(dots)) == 0
            return y.astype(np.float64), dots

        x, b = r.normal(size=(n, k)).astype(np.float32), r.normal(size=(n, k))
        D = r.uniform(1.0, 2.0, n).astype(np.float32)
        S32 = sp.csr_matrix((S.data.astype(np.float32).astype(np.float64), S.indices, S.indptr), shape=S.shape)
        x64, b32 = x.astype(np.float64), b.astype(np.float32)
        ax, size, ln = S32 @ x64, abs(S32) @ abs(x64), (np.diff(S.indptr) + 1)[:, None]
        err = ln * E32 * size + 1e-30
        y, _ = product(1, x, None, None)
        assert (abs(y - ax) <= err).all()
        for op, bb in ((2, b32), (4, b)):
            y, _ = product(op, x, bb, None)
            ref = b32 - ax
            assert (abs(y - ref) <= err + 2 * E32 * (abs(b32) + abs(ref) + err)).all()
        y, _ = product(3, x, b32, D)
        ref = (b32 - ax) / D[:, None] + x64
        mag = (abs(b32) + abs(ax) + err) / D[:, None] + abs(x64)
        assert (abs(y - ref) <= err / D[:, None] + 5 * E32 * mag).all()
        wr = r.normal(size=(2, n, k))
        y, dots = product(5, x, wr, None)
        ax, size = S @ x64, abs(S) @ abs(x64)
        assert (abs(y - ax) <= ln * E64 * size + 1e-300).all()
        for m, v in enumerate((wr[0], ax, wr[1])):
            lim = (n + 1) * E64 * (abs(v) * abs(x64)).sum(0) + (ln * E64 * size * abs(x64)).sum(0) + 1e-300
            assert (abs(dots[:, m] - (v * x64).sum(0)) <= lim).all()
        A.close()


def test_block_solve_follows_new_values(ctx):
    """A batched FP32-hierarchy solve on a matrix large enough for the block form, before and after
    its values change in place: the block copies follow."""
    n, row, col, val = bx.laplacian3d(27, 43, 41, 39)
    A = bx.CSR(ctx, n, n, row, col, val)
    S = sp.csr_matrix((val, col, row), shape=(n, n))
    p = bx.Params(solver="FCG", preconditioner="BCMG", precision="FP32", rtol=1e-9, prerelax_sweeps=1, postrelax_sweeps=1,
                  dispnorm=0)
    P = bx.prec_setup(ctx, A, p)
    B = np.random.default_rng(2).normal(size=(n, 16))
    for scale in (1.0, 3.0):
        A.update_values(val * scale)
        x, info = bx.solve(ctx, A, B, np.zeros((n, 16)), p, P)
        assert info["retv"] == 0
        R = B - scale * (S @ x)
        assert (np.linalg.norm(R, axis=0) <= 1.01e-9 * np.linalg.norm(B, axis=0)).all()
    P.finalize()
    A.close()
