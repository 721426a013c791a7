"""The Chebyshev preconditioner with several steps per launch on node tiles
(the device FEM system, which knows its node positions) against the same
solve with one step per launch (the sparse API, which does not): the same
products in the same order, so iterations, restarts and the solution agree
bit for bit.

Meshes at the edges of the tiles: smaller than one tile, one node over a
multiple of a wave, both tile sizes, rows wider than the uniform layout's
six blocks (the reference's tessellated meshes), node numbers in random
order, positions crowded into a corner (cells of very different counts) and
spread along one line of cells."""
import numpy as np
import pytest

from conftest import load_golden, problem_from_golden

pytestmark = pytest.mark.gpu


def _grid(nx, ny, jitter=0.0):
    from nbots_amd import synth
    p = synth.cantilever_traction(nx, ny)
    if jitter:
        p.nod = synth.grid(nx, ny, jitter=jitter)[0]
    return p


def _shuffled(nx, ny):
    p = _grid(nx, ny)
    new = np.random.default_rng(5).permutation(p.N_nod).astype(np.uint32)   # old -> new
    xy = np.empty((p.N_nod, 2))
    xy[new] = p.nod.reshape(-1, 2)
    p.nod = xy.reshape(-1)
    p.conn, p.vtx, p.sgm_nodes = new[p.conn], new[p.vtx], new[p.sgm_nodes]
    return p


def _crowded(nx, ny):
    p = _grid(nx, ny)
    q = p.nod.reshape(-1, 2) / np.array([nx, ny])
    p.nod = (q ** 3 * np.array([nx, ny]) + 0.02 * p.nod.reshape(-1, 2)).reshape(-1)
    return p


MESHES = {
    "below_a_tile_5x3": lambda: _grid(5, 3),
    "one_tile_15x9": lambda: _grid(15, 9),
    "64x32_jitter": lambda: _grid(64, 32, 0.1),
    "odd_131x67": lambda: _grid(131, 67),
    "slab_700x3": lambda: _grid(700, 3),
    "crowded_96x48": lambda: _crowded(96, 48),
    "shuffled_60x41": lambda: _shuffled(60, 41),
    "beam_mesh": lambda: problem_from_golden(load_golden("beam_cantilever")),
    "plate_mesh": lambda: problem_from_golden(load_golden("plate_with_hole")),
}


@pytest.mark.parametrize("degree", [2, 9, 40])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_tiles_equal_single_steps(mesh, degree):
    import nbots_amd as nb
    from nbots_amd.fem import Fem, SOLVE_MIXED, solve_opts
    p = MESHES[mesh]()
    o = solve_opts(cheb_degree=degree)
    f = Fem.from_problem(p)
    rp, col, val, F = f.system()
    A = nb.Sparse.from_csr(rp, col, val, vars_per_node=2)
    x, ia = A.solve(F, mode=SOLVE_MIXED, tol=1e-8, max_iter=20 * p.N, opts=o)
    i = f.solve(SOLVE_MIXED, tol=1e-8, opts=o)
    u = f.displacement()
    print(mesh, degree, i["iters"], i["layout"])
    assert i["status"] == ia["status"] == 0
    assert (i["iters"], i["outer"], i["fallback"]) == (ia["iters"], ia["outer"], ia["fallback"])
    assert np.array_equal(u, x)
    A.destroy()
    f.destroy()


@pytest.mark.parametrize("n", [(362, 181), (363, 181), (442, 220), (446, 220), (570, 287),
                               (811, 403), (810, 402)])
def test_tiles_equal_single_steps_at_the_rules_edges(n):
    """Around 65,536, 98,304, 163,840 and 327,680 nodes (tile counts, ring
    counts and the form of the rows' values): two outer iterations."""
    import nbots_amd as nb
    from nbots_amd.fem import Fem, SOLVE_MIXED
    p = _grid(*n)
    f = Fem.from_problem(p)
    rp, col, val, F = f.system()
    conn = p.conn.reshape(-1, 3).astype(np.int64)
    e = np.concatenate([conn[:, [0, 1]], conn[:, [1, 2]], conn[:, [2, 0]]])
    key = np.unique(np.concatenate([e, e[:, ::-1]]) @ np.array([p.N_nod, 1]))
    deg = np.bincount(key // p.N_nod, minlength=p.N_nod)
    A = nb.Sparse.from_graph(deg, np.split((key % p.N_nod).astype(np.uint32),
                                           np.cumsum(deg)[:-1]), vars_per_node=2)
    A.import_values(val)
    x, ia = A.solve(F, mode=SOLVE_MIXED, tol=1e-8, max_iter=2)
    i = f.solve(SOLVE_MIXED, tol=1e-8, max_iter=2)
    assert i["status"] == ia["status"] == 1 and i["iters"] == ia["iters"] == 2
    assert np.array_equal(f.displacement(), x)
    A.destroy()
    f.destroy()
