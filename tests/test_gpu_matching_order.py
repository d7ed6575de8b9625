"""The matching's preference order is total whatever the values: NaN weights come last and are never proposed to,
entries of one column and weight go by their place.  Against the sequential Suitor on the pairs that can be
proposed to: a pair's weight is that of its entry above the diagonal."""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchgx_amd as bx
import oracle_py as O

pytestmark = pytest.mark.gpu


def pairs(n, degree, seed):
    """random pairs above the diagonal, values with many ties"""
    r = np.random.default_rng(seed)
    U = sp.triu(sp.random(n, n, density=min(1.0, degree / n), random_state=r, format="csr"), 1).tocoo()
    return U.row, U.col, -r.integers(1, 6, len(U.row)) / 4.0, r


def assemble(n, i, j, v):
    """CSR arrays with the entries (i, j, v), those of one place kept apart in their order, and a diagonal"""
    i, j, v = np.concatenate([i, np.arange(n)]), np.concatenate([j, np.arange(n)]), np.concatenate([v, np.full(n, 30.0)])
    o = np.lexsort((np.arange(len(i)), j, i))
    row = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=n))]).astype(np.int32)
    return row, j[o].astype(np.int32), v[o]


@pytest.mark.parametrize("repeated", [False, True])
@pytest.mark.parametrize("n, degree", [(5, 3), (70, 3), (500, 8), (90, 60), (5000, 20), (140000, 4)])
def test_matching(ctx, n, degree, repeated):
    i, j, v, r = pairs(n, degree, n + degree)
    m = len(i)
    upper, lower = v.copy(), v.copy()
    nan = r.random(m) < 0.2
    upper[nan] = np.nan  # the weight of both
    lower[r.random(m) < 0.2] = np.nan  # not looked at
    ei, ej, ev = [i, j], [j, i], [upper, lower]
    if repeated:  # three entries in a place, the middle one of negative weight
        for u, l in ((np.ones(m), np.ones(m)), (upper, lower)):
            ei, ej, ev = ei + [i, j], ej + [j, i], ev + [u, l]
    A = bx.CSR(ctx, n, n, *assemble(n, np.concatenate(ei), np.concatenate(ej), np.concatenate(ev)))
    w = np.ones(n)
    M = A.matching(w)
    A.close()
    k = ~nan
    row, col, val = assemble(n, np.concatenate([i[k], j[k]]), np.concatenate([j[k], i[k]]), np.concatenate([v[k], v[k]]))
    assert np.array_equal(M, O.suitor(O.Csr.from_scipy(sp.csr_matrix((val, col, row), shape=(n, n))), w))


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
def test_nan_pair_is_an_error(ctx, precision):
    n, row, col, val = bx.laplacian3d(7, 9, 8, 7)
    S = sp.csr_matrix((val, col, row), shape=(n, n))
    S[100, 101] = S[101, 100] = np.nan
    A = bx.CSR.from_scipy(ctx, S)
    p = bx.Params(solver="FCG", preconditioner="BCMG", precision=precision, max_coarse_size=10, dispnorm=0)
    with pytest.raises(bx.BcmgxError, match="non-finite"):
        P = bx.prec_setup(ctx, A, p)
        bx.solve(ctx, A, np.ones(n), np.zeros(n), p, P)
    A.close()
