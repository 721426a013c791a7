"""Node rows of more blocks than the two-kernel Jacobi-PCG loads ahead (seven,
or three or four to either side of the diagonal): the rest is taken four at a
time (CgRow::product), so rows whose rest is one to five and many blocks, on the
symmetric copy and on full rows, against the oracle with the bars of the other
PCG tests."""
import numpy as np
import pytest

from test_gpu_pcg_two_kernels import _cut

pytestmark = pytest.mark.gpu


def _band(nodes, h, sym):
    """2x2 blocks to the h next nodes on either side in a ring"""
    rng = np.random.default_rng(11)
    c = np.sort((np.arange(nodes)[:, None] + np.arange(-h, h + 1)) % nodes, 1)
    row = np.repeat(np.arange(nodes), 2 * h + 1)
    a, b = np.minimum(row, c.ravel()), np.maximum(row, c.ravel())
    t = rng.uniform(-1.0, 1.0, (nodes, nodes, 2, 2))
    blk = np.where((row <= c.ravel())[:, None, None], t[a, b], t[a, b].transpose(0, 2, 1))
    d = np.flatnonzero(row == c.ravel())
    blk[d] = np.array([[1.0, 0.1], [0.1, 1.5]]) * (4.0 * h + 2.0)
    if not sym:
        blk[1, 0, 1] += 0.125
    rp = np.arange(2 * nodes + 1, dtype=np.uint32) * np.uint32(2 * (2 * h + 1))
    col = (2 * c[:, None, :, None] + np.arange(2)).repeat(2, 1)
    val = blk.reshape(nodes, 2 * h + 1, 2, 2).transpose(0, 2, 1, 3)
    return rp, col.astype(np.uint32).ravel(), np.ascontiguousarray(val).ravel()


@pytest.mark.parametrize("sym", [True, False])
@pytest.mark.parametrize("h", [3, 4, 5, 6, 8, 9, 25])
def test_wide_blocks(h, sym):
    import nbots_amd as nb
    rp, col, val = _band(330, h, sym)
    A = nb.Sparse.from_csr(rp, col, val, vars_per_node=2)
    assert A.is_blocked() == 1
    F = np.random.default_rng(5).standard_normal(660)
    _, info = A.solve(F, mode=0, tol=1e-30, max_iter=3)
    assert info["layout"] == int(sym)
    _cut(A, rp, col, val, F, n=3)
    _cut(A, rp, col, val, F, plain=True, n=3)
    A.destroy()
