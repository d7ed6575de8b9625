"""Rows that list a column twice: their entries add up in every product, so the block form (csrc/blocked.hip),
which has one place per row and column, is not made of them."""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu


def split(row, col, val, chosen, first=0.375):
    """the same operator with the chosen entries listed twice: first * value, then the rest of it"""
    times = 1 + chosen
    at = np.cumsum(times) - times  # an entry's place
    c, v = np.repeat(col, times), np.repeat(val, times)
    v[at[chosen]] *= first
    v[at[chosen] + 1] -= v[at[chosen]]
    return np.concatenate([[0], np.cumsum(times)])[row].astype(np.int32), c, v


@pytest.mark.parametrize("points, dims, entry", [(7, (2, 1, 1), 1), (27, (5, 4, 3), 0), (27, (5, 4, 3), -1), (27, (21, 19, 13), 5000)])
def test_block_form_refused(ctx, points, dims, entry):
    """one repeated entry: in the first, the last or an inner tile"""
    n, row, col, val = bx.laplacian3d(points, *dims)
    chosen = np.zeros(len(val), bool)
    chosen[entry] = True
    r2, c2, v2 = split(row, col, val, chosen)
    k, order = 8, np.arange(n, dtype=np.int32)
    x, y, dots = np.ones((n, k), np.float32), np.zeros((n, k), np.float32), np.zeros((k, 3))
    p = lambda v: v.ctypes.data_as(bx.C.c_void_p)
    for arrays, refused in (((row, col, val), False), ((r2, c2, v2), True)):
        A = bx.CSR(ctx, n, n, *arrays)
        code = bx.lib().bcmgx_internal_block_product(ctx.h, A.h, p(order), k, 1, p(x), None, None, p(y), p(dots))
        assert (code != 0) == refused
        A.close()


@pytest.mark.parametrize("k", [7, 16])
def test_solve(ctx, k):
    """a batched solve with an FP32 hierarchy, twice (launched, then replayed), on a matrix large enough for the
    block form: the solution is that of the summed matrix.  Bound: the solver's own, 1 % more for its recurrence."""
    n, row, col, val = bx.laplacian3d(27, 43, 41, 39)
    r = np.repeat(np.arange(n), np.diff(row))
    chosen = (r != col) & ((r + col) % 5 == 0)  # both entries of a pair
    A = bx.CSR(ctx, n, n, *split(row, col, val, chosen))
    S = sp.csr_matrix((val, col, row), shape=(n, n))
    p = bx.Params(solver="FCG", preconditioner="BCMG", precision="FP32", rtol=1e-9, prerelax_sweeps=1, postrelax_sweeps=1,
                  dispnorm=0)
    P = bx.prec_setup(ctx, A, p)
    for seed in (1, 2):
        B = np.random.default_rng(seed).normal(size=(n, k))
        x, info = bx.solve(ctx, A, B, np.zeros((n, k)), p, P)
        assert info["retv"] == 0
        assert (np.linalg.norm(B - S @ x, axis=0) <= 1.01e-9 * np.linalg.norm(B, axis=0)).all()
    P.finalize()
    A.close()
