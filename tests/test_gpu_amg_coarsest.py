"""The coarsest level's inverse on the device (k_dense_sweep).

A system of at most 200 unknowns is its own coarsest level, so its
preconditioner is that inverse alone, in FP32: the flexible CG then needs at
most 3 iterations to 1e-8 (each reduces the error by about the inverse's
accuracy, 1e-7 times the condition number of at most 1e5), whatever the
number of entries a thread holds (1 to 7 squared: the sizes below, with the
edges of 32, 64, ... unknowns that these meshes reach).  The displacement
agrees with an FP64 solve within rel-L2 1e-6, the bar of the other AMG
solves.  Unknowns that a singular matrix leaves without a pivot are dropped:
a second body without supports or loads stays at rest."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(p):
    from nbots_amd.fem import Fem, MIXED_AMG_FCG, SOLVE_FP64, SOLVE_MIXED, solve_opts
    f, g = Fem.from_problem(p), Fem.from_problem(p)
    ia = f.solve(SOLVE_MIXED, tol=1e-8, max_iter=50, opts=solve_opts(MIXED_AMG_FCG))
    i64 = g.solve(SOLVE_FP64, tol=1e-11)
    u, v = f.displacement(), g.displacement()
    f.destroy()
    g.destroy()
    assert ia["status"] == 0 and i64["status"] == 0, (ia, i64)
    return ia, u, v


@pytest.mark.parametrize("nx,ny", [(1, 1), (3, 3), (7, 1), (7, 3), (10, 2), (11, 3), (15, 3),
                                   (12, 4), (15, 4), (11, 7), (9, 9)])
def test_dense_alone(nx, ny):
    """8, 32, 32, 64, 66, 96, 128, 130, 160, 192 and 200 unknowns"""
    from nbots_amd import synth
    p = synth.cantilever_traction(nx, ny, seed=3, sigma=0.5)
    print(f"[amg coarsest] {nx}x{ny}: {p.N}", flush=True)
    ia, u, v = _solve(p)
    assert ia["iters"] <= 3 and not ia["layout"] & 2, ia
    assert np.linalg.norm(u - v) <= 1e-6 * np.linalg.norm(v)


def test_unknowns_without_a_pivot():
    from nbots_amd import synth
    a, b = synth.cantilever_traction(5, 3, seed=3, sigma=0.5), synth.cantilever_traction(4, 2, seed=4)
    nod = np.concatenate([a.nod, b.nod + 100.0])
    conn = np.concatenate([a.conn, b.conn + np.uint32(a.N_nod)]).astype(np.uint32)
    p = dataclasses.replace(a, nod=nod, conn=conn,
                            elem_E=np.concatenate([a.elem_E, b.elem_E]))
    print(f"[amg coarsest] two bodies: {p.N}", flush=True)
    ia, u, v = _solve(p)
    assert ia["iters"] <= 3, ia
    assert np.linalg.norm(u - v) <= 1e-6 * np.linalg.norm(v)
    assert np.all(u[a.N:] == 0.0)
