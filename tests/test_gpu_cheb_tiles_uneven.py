"""Meshes on which tiles of several Chebyshev steps per launch do not pay (or
that outgrow them) take a step per launch: an outer iteration of the device
system is no slower than the sparse API's on the same matrix, which knows no
node positions and never has tiles (20 % for the spread of the timings), and its
result is the same to the bit.

Spacing that grows along one side, an unstructured mesh of even density with
more than 512 * 528 nodes (rows of up to eleven blocks), and a large mesh whose
nodes are numbered in random order (15 % there: it took 24 % longer)."""
import numpy as np
import pytest

from test_gpu_amg_bottom import delaunay
from test_gpu_cheb_tiles import _shuffled

pytestmark = pytest.mark.gpu


def _graded(nx, ny):
    """Four fifths of the rows of nodes in the lowest fifth of the height"""
    from nbots_amd import synth
    p = synth.cantilever_traction(nx, ny)
    q = p.nod.reshape(-1, 2).copy()
    t = q[:, 1] / ny
    q[:, 1] = ny * np.where(t < 0.8, 0.25 * t, 0.2 + 4.0 * (t - 0.8))
    p.nod = q.reshape(-1)
    return p


MESHES = {"graded": _graded, "delaunay": delaunay, "shuffled": _shuffled}


@pytest.mark.parametrize("kind,nx,ny,bar", [("graded", 724, 362, 1.2), ("delaunay", 740, 370, 1.2),
                                            ("shuffled", 1430, 720, 1.15)])
def test_no_slower_than_single_steps(kind, nx, ny, bar):
    import nbots_amd as nb
    from nbots_amd.fem import Fem, SOLVE_MIXED
    p = MESHES[kind](nx, ny)
    f = Fem.from_problem(p)
    rp, col, val, F = f.system()
    conn = p.conn.reshape(-1, 3).astype(np.int64)
    e = np.concatenate([conn[:, [0, 1]], conn[:, [1, 2]], conn[:, [2, 0]]])
    key = np.unique(np.concatenate([e, e[:, ::-1]]) @ np.array([p.N_nod, 1]))
    deg = np.bincount(key // p.N_nod, minlength=p.N_nod)
    A = nb.Sparse.from_graph(deg, np.split((key % p.N_nod).astype(np.uint32),
                                           np.cumsum(deg)[:-1]), vars_per_node=2)
    A.import_values(val)
    ms = [np.inf, np.inf]
    for _ in range(3):
        x, ia = A.solve(F, mode=SOLVE_MIXED, tol=1e-14, max_iter=8)
        i = f.solve(SOLVE_MIXED, tol=1e-14, max_iter=8)
        assert i["iters"] == ia["iters"] == 8
        ms = [min(ms[0], ia["ms"]), min(ms[1], i["ms"])]
    print(kind, [1e3 * m / 8 for m in ms])
    assert np.array_equal(f.displacement(), x)
    assert ms[1] <= bar * ms[0]
    A.destroy()
    f.destroy()


def test_first_solve_of_a_crowded_mesh():
    """Four fifths of the nodes in a 400th of the area, where no attempt fits:
    finding that out takes the first solve no longer than cutting the even mesh
    does (twice its time for the spread)."""
    import time

    from nbots_amd import synth
    from nbots_amd.fem import Fem, SOLVE_MIXED
    nx, ny = 1024, 512
    best = {}
    for even in (True, False, True, False):
        p = synth.cantilever_traction(nx, ny)
        if not even:
            t = p.nod.reshape(-1, 2) / np.array([nx, ny])
            t = np.where(t < 0.8, 0.0625 * t, 0.05 + 4.75 * (t - 0.8))
            p.nod = (t * np.array([nx, ny])).reshape(-1)
        f = Fem.from_problem(p)
        t0 = time.perf_counter()
        f.solve(SOLVE_MIXED, tol=1e-14, max_iter=1)
        best[even] = min(best.get(even, np.inf), time.perf_counter() - t0)
        f.destroy()
    print(best)
    assert best[False] <= 2.0 * best[True]
