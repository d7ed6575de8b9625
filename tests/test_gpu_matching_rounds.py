"""The matching's rounds (csrc/setup.hip) against the sequential Suitor: the matching of a total order is
unique, so equal entries.  131072 vertices (4 lanes each, 256 CUs of 2048 threads) are matched in one
round and more in two or several; lists of 0, 1 and more than 4 candidates; ties everywhere and nowhere."""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchgx_amd as bx
import oracle_py as O

pytestmark = pytest.mark.gpu


def grid(points, dims, weights):
    n, row, col, val = bx.laplacian3d(points, *dims)
    S = sp.csr_matrix((val, col, row), shape=(n, n))
    if weights:
        U = sp.triu(S, 1).tocsr()
        U.data = -np.random.default_rng(n).uniform(0.5, 2.0, U.nnz)
        S = (U + U.T + sp.diags(np.full(n, 30.0))).tocsr()
        S.sort_indices()
    return S


@pytest.mark.parametrize("weights", [False, True])
@pytest.mark.parametrize("points, dims", [(7, (1, 1, 1)), (7, (2, 1, 1)), (7, (3, 1, 1)), (27, (2, 2, 2)), (7, (64, 64, 32)),
                                          (27, (51, 51, 51)), (7, (131, 91, 11)), (27, (67, 65, 61))])
def test_matching(ctx, points, dims, weights):
    S = grid(points, dims, weights)
    A = bx.CSR.from_scipy(ctx, S)
    n = S.shape[0]
    w = np.random.default_rng(1).uniform(0.5, 2.0, n) if weights else np.ones(n)
    assert np.array_equal(A.matching(w), O.suitor(O.Csr.from_scipy(S), w))
    A.close()
