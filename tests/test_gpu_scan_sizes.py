"""The exclusive scan's forms (csrc/prims.hip) at their edges, through a transpose: the row pointers of the
transpose are the scan of the column counts.  Exact."""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu


# one workgroup (1024 items a turn, to 4096), blocks that sum the totals before them (to 1024 blocks of 1024), three launches
@pytest.mark.parametrize("m", [1, 1023, 1024, 1025, 4095, 4096, 4097, 5121, 263000, 1 << 20, (1 << 20) + 1, 3000001])
def test_transpose_row_pointers(ctx, m):
    r = np.random.default_rng(m)
    n, per = 500, min(m, 40)
    col = np.concatenate([np.sort(r.choice(m, size=per, replace=False)) if m < 10000 else np.unique(r.integers(0, m, size=per)) for _ in range(n - 1)] + [[m - 1]])
    ptr = np.linspace(0, len(col), n + 1).astype(np.int32)
    S = sp.csr_matrix((r.normal(size=len(col)), col.astype(np.int32), ptr), shape=(n, m))
    S.sum_duplicates()
    A = bx.CSR.from_scipy(ctx, S)
    T = A.transpose().to_scipy()
    assert np.array_equal(T.indptr, S.T.tocsr().indptr)
    assert (T != S.T.tocsr()).nnz == 0
    A.close()
