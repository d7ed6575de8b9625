"""The column-table kernel of the AFSAI setup (csrc/afsai.hip) against the oracle, where its
bookkeeping changes: pattern sizes around 16 (the system's second part), rows that bring 30 and 31
entries into the table, tables near their limit, rows handed to the merge beside rows that are not,
breakdowns, row counts that leave groups of the last wave empty.

The factor's pattern must be the oracle's; its values agree to 1e-12 (the operations and their order
are the oracle's, the square roots and divisions correctly rounded on both sides)."""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchgx_amd as bx
import oracle_py as O

pytestmark = pytest.mark.gpu


def banded(n, offsets, rng):
    """SPD, symmetric to the bit, entries on the given diagonals."""
    d = {o: rng.uniform(-1.0, -0.1, n - o) for o in offsets}
    S = sp.diags([d[o] for o in offsets], list(offsets), shape=(n, n))
    S = S + S.T
    S = S + sp.diags(np.asarray(abs(S).sum(axis=1)).ravel() * 1.02 + 1e-3)
    S = S.tocsr()
    S.sort_indices()
    return S


CASES = {
    "tridiagonal": lambda r: banded(67, (1,), r),
    "one_row": lambda r: sp.csr_matrix(np.array([[3.0]])),
    "five_rows": lambda r: banded(5, (1, 2, 3), r),
    "left_30": lambda r: banded(300, tuple(range(1, 31)), r),
    "left_31": lambda r: banded(301, tuple(range(1, 32)), r),
    "left_33": lambda r: banded(302, tuple(range(1, 34)), r),
    "wide_table": lambda r: banded(900, (1, 2, 3, 5, 8, 13, 21, 34, 55, 89, 144, 233), r),
    "seven_point": lambda r: banded(11 * 10 * 9, (1, 11, 110), r),
    "mixed_rows": lambda r: sp.block_diag([banded(130, tuple(range(1, 40)), r), banded(131, (1, 7), r)]).tocsr(),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_afsai_factor(ctx, name):
    S = CASES[name](np.random.default_rng(len(name)))
    p = bx.Params(preconditioner="AFSAI", dispnorm=0)
    A = bx.CSR.from_scipy(ctx, S)
    P = bx.prec_setup(ctx, A, p)
    G = P.afsai_factor()
    o = O.Prec(O.Csr.from_scipy(S), p.s).afsai_G().to_scipy()
    assert np.array_equal(G.indptr, o.indptr) and np.array_equal(G.indices, o.indices)
    assert np.abs(G.data - o.data).max() <= 1e-12 * np.abs(o.data).max()
    P.finalize()
    A.close()
