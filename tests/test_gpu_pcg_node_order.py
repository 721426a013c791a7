"""The limit of the two-kernel Jacobi-PCG for rows that are not three and three
blocks to either side of the diagonal (131,072 nodes): nodes numbered in random
order.  Just below the limit the cut solve agrees with the oracle as the other
limits do; and a size near the limit of ordered meshes, 196,608 nodes, takes no
more than a tenth longer per iteration than one just above, where there are
five kernels in any case."""
import numpy as np
import pytest

from test_gpu_cheb_tiles import _shuffled
from test_gpu_pcg_two_kernels import _system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(361, 361), (362, 361)])
def test_shuffled_limits(n):
    """131,044 nodes (two kernels) and 131,406 (five)"""
    import oracle
    from nbots_amd.fem import Fem, SOLVE_REFERENCE
    p = _shuffled(*n)
    rp, col, val, F = _system(p)
    ref = oracle.pcg(rp, col, val, F, max_iter=7, tol=1e-30)
    f = Fem.from_problem(p)
    i = f.solve(SOLVE_REFERENCE, tol=1e-30, max_iter=7)
    assert (i["status"], i["iters"], i["layout"]) == (1, 7, 1)
    assert abs(i["tol_reached"] - ref[2]) <= 1e-9 * ref[2]
    u = f.displacement()
    assert np.linalg.norm(u - ref[0]) <= 1e-11 * np.linalg.norm(ref[0])
    f.destroy()


def test_shuffled_is_no_slower_below_the_limit_of_ordered_meshes():
    from nbots_amd.fem import Fem, SOLVE_FP64
    us = []
    for n in ((442, 442), (443, 443)):
        f = Fem.from_problem(_shuffled(*n))
        best = np.inf
        for _ in range(3):
            i = f.solve(SOLVE_FP64, tol=1e-13, max_iter=256)
            best = min(best, i["ms"] / i["iters"])
        us.append(1e3 * best)
        f.destroy()
    print(us)
    assert us[0] <= 1.1 * us[1]
