"""Scalar CSR rows of many entries in the two-kernel Jacobi-PCG, which takes
them a strip of every row at a time (k_cg_dir_csr): row lengths around a
multiple of a strip, rows of different lengths in one workgroup, a last
workgroup of few rows, and both sides of the rule (64 entries a row on
average, the longest of at most a sixteenth of the workgroup's entries) against
the oracle: tol_reached within 1e-9 relative and x within rel-L2 1e-11, the
bars of the other PCG tests."""
import numpy as np
import pytest

from test_gpu_pcg_two_kernels import _cut, _laplacian

pytestmark = pytest.mark.gpu


def _band(n, h):
    """h neighbours to either side of each of n nodes in a ring"""
    off = np.concatenate([np.arange(-h, 0), np.arange(1, h + 1)])
    return list(np.sort((np.arange(n)[:, None] + off) % n, 1).astype(np.uint32))


def _random(n, mean, hub=0):
    """Symmetric adjacency of about `mean` neighbours, between a few and many;
    node 3 has `hub` more."""
    rng = np.random.default_rng(7)
    a = rng.random((n, n)) < np.outer(*2 * [rng.uniform(0.3, 1.7, n)]) * mean / n
    a[3, :hub] = True
    a |= a.T
    np.fill_diagonal(a, False)
    return [np.flatnonzero(r).astype(np.uint32) for r in a]


CASES = {
    "63": lambda: _band(256, 31),             # below the rule: tiles
    "65_one_row_over": lambda: _band(257, 32),
    "71": lambda: _band(300, 35),
    "73": lambda: _band(300, 36),
    "dense": lambda: _band(301, 150),
    "uneven": lambda: _random(700, 90),
    "one_too_long": lambda: _random(1500, 40, hub=1499),
}


@pytest.mark.parametrize("case", list(CASES))
def test_long_rows(case):
    rng = np.random.default_rng(3)
    A, rp, col, val = _laplacian(CASES[case](), 1, rng)
    assert A.is_blocked() == 0
    b = rng.standard_normal(rp.size - 1)
    # (three iterations: systems this dense converge by a factor of ten in each)
    _cut(A, rp, col, val, b, n=3)
    _cut(A, rp, col, val, b, plain=True, n=3)
    A.destroy()


def test_time_grows_no_faster_than_the_entries():
    """2,001 rows of 33 entries and of 513: an iteration of the second system
    takes no more than 513 / 33 times as long."""
    rng = np.random.default_rng(3)
    us = []
    for h in (16, 256):
        A, rp, col, val = _laplacian(_band(2001, h), 1, rng)
        b = rng.standard_normal(2001)
        best = np.inf
        for _ in range(3):
            _, i = A.solve(b, mode=0, tol=1e-300, max_iter=64)
            best = min(best, i["ms"] / i["iters"])
        us.append(1e3 * best)
        A.destroy()
    print(us)
    assert us[1] <= 513 / 33 * us[0]
