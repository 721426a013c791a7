"""The product with the symmetric copy (indexes of both parts loaded first,
places from one slice width where there is one) against the full layout and the
oracle's row sums, bit for bit: banded patterns, whose slices all have one
width, with rows of fewer, as many and more blocks than a batch of three or
four, and a pattern of uneven rows, which keeps its slice offsets.  One system
beyond the two-kernel PCG, whose five kernels read the copy through the caches
four blocks at a time, against the same five iterations in numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _blocks(n, half, rng, uneven=False):
    """CSR of a symmetric matrix of 2x2 blocks with `half` upper blocks a row
    (uneven: three, and fifteen on every 61st)."""
    import scipy.sparse as sp
    reach = np.full(n, half)
    if uneven:
        reach[::61] = 15
    i = np.repeat(np.arange(n), reach)
    j = i + 1 + np.concatenate([np.arange(r) for r in reach]) if len(i) else i
    i, j = i[j < n], j[j < n]
    B = rng.standard_normal((len(i), 2, 2))
    D = rng.standard_normal((n, 2, 2))
    D = D + D.transpose(0, 2, 1) + (8.0 + 8.0 * (15 if uneven else half)) * np.eye(2)
    r = np.concatenate([i, j, np.arange(n)])
    c = np.concatenate([j, i, np.arange(n)])
    v = np.concatenate([B, B.transpose(0, 2, 1), D])
    o = np.lexsort((c, r))
    ptr = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))])
    A = sp.bsr_matrix((v[o], c[o], ptr), shape=(2 * n, 2 * n)).tocsr()
    A.sort_indices()
    return A


@pytest.mark.parametrize("n,half,uneven", [
    (1, 1, False), (64, 1, False), (65, 2, False), (257, 3, False), (1000, 4, False),
    (1027, 5, False), (2000, 6, False), (2001, 8, False), (2050, 9, False), (3001, 3, True)])
def test_rows_bit_exact(n, half, uneven):
    import nbots_amd as nb
    import oracle
    rng = np.random.default_rng(n + half)
    S = _blocks(n, half, rng, uneven)
    rp, col = S.indptr.astype(np.uint32), S.indices.astype(np.uint32)
    A = nb.Sparse.from_csr(rp, col, S.data, vars_per_node=2)
    x = rng.standard_normal(2 * n)
    full = A.matvec(x)
    _, info = A.solve(rng.standard_normal(2 * n), mode=1, tol=1e-6)
    assert info["layout"] == 1 and info["status"] == 0
    sym = A.matvec(x)
    assert np.array_equal(sym, full)
    assert np.array_equal(sym, oracle.spmv(rp, col, S.data, x))
    A.destroy()


@pytest.mark.parametrize("half", [2, 5])
def test_five_kernel_pcg_through_the_caches(half):
    import nbots_amd as nb
    n = 196_700
    rng = np.random.default_rng(half)
    S = _blocks(n, half, rng)
    b = rng.standard_normal(2 * n)
    A = nb.Sparse.from_csr(S.indptr.astype(np.uint32), S.indices.astype(np.uint32), S.data,
                           vars_per_node=2)
    x, info = A.solve(b, mode=1, tol=1e-30, max_iter=5)
    assert info["layout"] == 1 and info["iters"] == 5
    d, y = S.diagonal(), np.zeros(2 * n)
    g = -b
    q = g / d
    p, rz = -q, g @ q
    for _ in range(5):
        w = S @ p
        a = rz / (p @ w)
        y += a * p
        g = g + a * w
        q = g / d
        rz, old = g @ q, rz
        p = -q + (rz / old) * p
    # sums of 4e5 terms in other orders: relative differences of 1e-13 a
    # scalar, five times over, on a well conditioned matrix
    assert np.linalg.norm(x - y) <= 1e-10 * np.linalg.norm(y)
    A.destroy()
