"""bcmgx_spmm on device columns in place (csrc/tiled.hip and the one-column kernels) against the staged
products of the same matrix: equal bits, for every operation.

Both sum a row in CSR order with the product and the sum rounded apart (k > 1), or run the same kernel
(k = 1), so no tolerance is needed.
"""
import numpy as np
import pytest
import scipy.sparse as sp

import bootcmatchgx_amd as bx

pytestmark = pytest.mark.gpu


def lap(points, *dims):
    n, row, col, val = bx.laplacian3d(points, *dims)
    return sp.csr_matrix((val, col, row), shape=(n, n))


def strips(n, width, seed, m=None, reverse=False):
    """row i: `width` consecutive columns from width * i (mod m): 64 * width distinct ones a tile"""
    m = m or n
    r = np.random.default_rng(seed)
    col = (np.arange(n)[:, None] * width + np.arange(width)) % m
    col = -np.sort(-col, 1) if reverse else np.sort(col, 1)
    S = sp.csr_matrix((r.normal(size=n * width), col.ravel(), np.arange(n + 1) * width), shape=(n, m))
    return S


def gaps():
    """rows of 0 to 8 entries, a tile without any, a last tile of one row"""
    n = 64 * 3 + 1
    length = np.arange(n) % 9
    length[64:128] = 0
    ptr = np.concatenate([[0], np.cumsum(length)])
    col = np.concatenate([min(i, n - 9) + np.arange(l) for i, l in enumerate(length)]).astype(np.int32)
    return sp.csr_matrix((np.random.default_rng(2).normal(size=ptr[-1]), col, ptr), shape=(n, n))


# tiles of 1, 63 to 65 rows; up to 639, 640 and 1024 distinct columns; rows of 8, 28 and 32 entries
MATRICES = {
    "one": lambda: sp.csr_matrix(np.array([[2.5]])),
    "grid7": lambda: lap(7, 63, 11, 5),
    "grid27": lambda: lap(27, 65, 13, 7),
    "grid27_thin": lambda: lap(27, 5, 3, 1),
    "u576": lambda: strips(64 * 5, 9, 3, 4000),
    "u640": lambda: strips(64 * 4 + 3, 10, 4, 3001, reverse=True),
    "u1024": lambda: strips(64 * 4 + 63, 16, 5, 4096),
    "wide28": lambda: strips(130, 28, 6, 700),
    "wide32": lambda: strips(130, 32, 7, 900),
    "gaps": gaps,
    "short_runs": lambda: sp.random(300, 300, 0.02, format="csr", random_state=8),
}
OPS = [(1, 1.0, 0.0), (2, -1.0, 1.0), (0, 0.7, -1.3)]


def block(ctx, host):
    d = bx.DeviceArray(ctx, (host.size,))
    d.upload(np.ascontiguousarray(host).ravel())
    return d


@pytest.mark.parametrize("k", [1, 2, 5, 8, 9, 31, 64])
@pytest.mark.parametrize("name", sorted(MATRICES))
def test_in_place_matches_staged(ctx, name, k):
    S = MATRICES[name]()
    A = bx.CSR.from_scipy(ctx, S) if S.has_sorted_indices else bx.CSR(ctx, S.shape[0], S.shape[1], S.indptr, S.indices, S.data)
    A.analyse()
    n, m = S.shape
    r = np.random.default_rng(k)
    X, Y = r.normal(size=(m, k)), r.normal(size=(n, k))
    X[m // 2, 0] = np.inf
    X[m // 3, k - 1] = np.nan
    ld = max(n, m) + 3
    for op, al, be in OPS:
        want = A.spmm(X, Y, al, be, op)
        x, y = np.full((k, ld), 7.0), np.full((k, ld), 9.0)
        x[:, :m], y[:, :n] = X.T, Y.T
        dx, dy = block(ctx, x), block(ctx, y)
        A.spmm_device(dx.ptr, dy.ptr, k, ld, al, be, op)
        got = dy.download().reshape(k, ld)
        assert np.array_equal(got[:, :n].T, want, equal_nan=True), op
        assert np.all(got[:, n:] == 9.0)
    A.close()


def test_overlapping_columns_are_staged(ctx):
    S = lap(7, 30, 20, 10)
    n, k = S.shape[0], 3
    A = bx.CSR.from_scipy(ctx, S)
    A.analyse()
    X = np.random.default_rng(1).normal(size=(n, k))
    want = A.spmm(X)
    for cols in (k, 1):
        b = block(ctx, X.T[:cols])
        A.spmm_device(b.ptr, b.ptr, cols, n)
        assert np.array_equal(b.download().reshape(cols, n).T, A.spmm(X[:, :cols]) if cols == 1 else want)
    A.close()
