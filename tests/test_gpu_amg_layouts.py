"""The multigrid levels' block layouts on the GPU: one width for all slices
where that adds little or the level is small, a width per slice otherwise.

Meshes with a hub, a node of some sixty neighbours whose aggregate is several
times as wide as any other: on the small one every layout has one width and
most of it padding, on the large one P^T of the finest level keeps a width
per slice.  A wrong block shows as extra
iterations: no solve may take more than the same cycle took with a width per
slice on every level (46, and 70 with five restarts of the flexible CG's
direction), and its displacement agrees with an FP64 solve within rel-L2
1e-6."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def hub(nx, ny, spokes=60):
    """The nx x ny cantilever's nodes, but around the middle a hub within a
    ring of `spokes` nodes, triangulated anew."""
    from scipy.spatial import Delaunay
    from nbots_amd import synth
    p = synth.cantilever_point(nx, ny, jitter=0.0)
    nod = p.nod.reshape(-1, 2).copy()
    c = np.array([nx / 2 + 0.25, ny / 2 + 0.25])
    inner = (nod[:, 0] > 0) & (nod[:, 0] < nx) & (nod[:, 1] > 0) & (nod[:, 1] < ny)
    nod[inner] += np.random.default_rng(3).uniform(-.2, .2, (inner.sum(), 2))
    near = np.flatnonzero(inner & (np.hypot(*(nod - c).T) < 5.0))
    ang = 2 * np.pi * np.arange(spokes) / spokes
    # the nodes near the middle move to the hub and the ring; the ones left
    # over take the places behind the ring's
    put = np.concatenate([[c], c + 4.0 * np.c_[np.cos(ang), np.sin(ang)],
                          c + 4.6 * np.c_[np.cos(ang), np.sin(ang)]])
    assert near.size <= len(put) and near.size > spokes
    nod[near] = put[:near.size]
    t = Delaunay(nod).simplices
    a, b, d = (nod[t[:, k]] for k in range(3))
    area = (b[:, 0] - a[:, 0]) * (d[:, 1] - a[:, 1]) - (d[:, 0] - a[:, 0]) * (b[:, 1] - a[:, 1])
    t, area = t[np.abs(area) > 1e-6], area[np.abs(area) > 1e-6]
    t[area < 0] = t[area < 0][:, [0, 2, 1]]
    return dataclasses.replace(p, nod=nod.ravel(), conn=t.astype(np.uint32).ravel())


@pytest.mark.parametrize("nx,ny,count", [(48, 24, 46), (192, 96, 70)])
def test_amg_layouts(nx, ny, count):
    from nbots_amd.fem import Fem, MIXED_AMG_FCG, SOLVE_FP64, SOLVE_MIXED, solve_opts
    p = hub(nx, ny)
    f, g = Fem.from_problem(p), Fem.from_problem(p)
    print(f"[amg layouts] {nx}x{ny}", flush=True)
    ia = f.solve(SOLVE_MIXED, tol=1e-8, max_iter=500,
                 opts=solve_opts(MIXED_AMG_FCG, true_residual=True))
    i64 = g.solve(SOLVE_FP64, tol=1e-11, opts=solve_opts(true_residual=True))
    ua, u64 = f.displacement(), g.displacement()
    f.destroy()
    g.destroy()
    print(ia["iters"], count, np.linalg.norm(ua - u64) / np.linalg.norm(u64))
    assert ia["status"] == 0 and i64["status"] == 0, (ia, i64)
    assert ia["iters"] <= count, ia
    assert np.linalg.norm(ua - u64) <= 1e-6 * np.linalg.norm(u64)
