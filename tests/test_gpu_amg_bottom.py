"""The last smoothed level and the dense solve below it in one workgroup
(k_amg_bottom), on the GPU.

Meshes whose last smoothed level takes each form of the kernel, and the ones
just beyond it that keep a launch per step (unknowns and widest block row of
that level in the parameters).  An error in the cycle's bottom shows as extra
iterations: each solve may take three more than the FP64 mirror of the same
hierarchy on the CPU (tests/amg/amg_host_check.cpp, the counts below; the
margin of the other AMG solves: the V-cycle is FP32 with an fp16 copy of the
finest off-diagonal blocks), and its displacement agrees with an FP64 solve
within rel-L2 1e-6, the bar of the other AMG solves."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def delaunay(nx, ny):
    """The nx x ny cantilever's nodes moved by up to 0.45 and triangulated
    anew: rows of up to 11 blocks, coarse ones of up to 20."""
    from scipy.spatial import Delaunay
    from nbots_amd import synth
    p = synth.cantilever_point(nx, ny, jitter=0.0)
    nod = p.nod.reshape(-1, 2).copy()
    inner = (nod[:, 0] > 0) & (nod[:, 0] < nx) & (nod[:, 1] > 0) & (nod[:, 1] < ny)
    nod[inner] += np.random.default_rng(3).uniform(-.45, .45, (inner.sum(), 2))
    t = Delaunay(nod).simplices
    a, b, c = (nod[t[:, k]] for k in range(3))
    area = (b[:, 0] - a[:, 0]) * (c[:, 1] - a[:, 1]) - (c[:, 0] - a[:, 0]) * (b[:, 1] - a[:, 1])
    t, area = t[np.abs(area) > 1e-6], area[np.abs(area) > 1e-6]
    t[area < 0] = t[area < 0][:, [0, 2, 1]]
    return dataclasses.replace(p, nod=nod.ravel(), conn=t.astype(np.uint32).ravel())


def mesh(kind, nx, ny):
    from nbots_amd import synth
    return delaunay(nx, ny) if kind == "delaunay" else synth.cantilever_point(nx, ny)


# mesh, outer iterations of the mirror to a true relative residual of 1e-8
CASES = [
    ("grid", 34, 17, 21),        # 216 unknowns, 11 blocks: one row per thread
    ("grid", 54, 27, 22),        # 540: two rows, the second of 28 threads
    ("grid", 76, 38, 22),        # 1,014: two rows of almost every thread
    ("grid", 77, 39, 22),        # 1,092: beyond, a launch per step
    ("delaunay", 40, 20, 21),    # 330, 17 blocks: one long row per thread
    ("delaunay", 64, 32, 22),    # 807, 20 blocks: beyond
    ("delaunay", 128, 64, 24),   # 201, 19 blocks, two smoothed levels above
]


@pytest.mark.parametrize("kind,nx,ny,mirror", CASES)
def test_amg_bottom_forms(kind, nx, ny, mirror):
    from nbots_amd.fem import Fem, MIXED_AMG_FCG, SOLVE_FP64, SOLVE_MIXED, solve_opts
    p = mesh(kind, nx, ny)
    f, g = Fem.from_problem(p), Fem.from_problem(p)
    print(f"[amg bottom] {kind} {nx}x{ny}", flush=True)
    ia = f.solve(SOLVE_MIXED, tol=1e-8, max_iter=500,
                 opts=solve_opts(MIXED_AMG_FCG, true_residual=True))
    i64 = g.solve(SOLVE_FP64, tol=1e-11, opts=solve_opts(true_residual=True))
    ua, u64 = f.displacement(), g.displacement()
    f.destroy()
    g.destroy()
    print(ia["iters"], mirror, np.linalg.norm(ua - u64) / np.linalg.norm(u64))
    assert ia["status"] == 0 and i64["status"] == 0, (ia, i64)
    assert ia["iters"] <= mirror + 3, ia
    assert np.linalg.norm(ua - u64) <= 1e-6 * np.linalg.norm(u64)
