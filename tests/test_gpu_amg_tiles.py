"""Levels between the finest and the bottom, smoothed on tiles in two launches
per cycle (k_amg_down, k_amg_up), on the GPU.

Meshes whose middle levels take each form of the kernels (tiles of up to 170
and of up to 341 block rows, rows of up to 14 and of up to 24 blocks, sums by
two and by four lanes, degrees 2, 4 and 5), one cut into a single line of
cells, and one of a level below the smallest that is tiled.  An error in a
cycle shows as extra iterations: each solve may take three more than the FP64
mirror of the same hierarchy on the CPU (tests/amg/amg_host_check.cpp, the
counts below; the V-cycle is FP32 with an fp16 copy of the finest off-diagonal
blocks) and reaches its tolerance in the true residual."""
import numpy as np
import pytest

from test_gpu_amg_bottom import mesh

pytestmark = pytest.mark.gpu

CASES = [
    ("grid", 96, 48, 22),        # 544 block rows, degree 2, four lanes
    ("grid", 333, 12, 26),       # 555, two lanes; 74 of degree 4 in one workgroup
    ("grid", 448, 224, 29),      # 11,250 in tiles of 200; 962 of degree 4
    ("delaunay", 128, 64, 24),   # 1,022 of up to 19 blocks
    ("grid", 34, 17, 21),        # none
]


@pytest.mark.parametrize("kind,nx,ny,mirror", CASES)
def test_amg_tiled_levels(kind, nx, ny, mirror):
    from nbots_amd.fem import Fem, MIXED_AMG_FCG, SOLVE_MIXED, solve_opts
    p = mesh(kind, nx, ny)
    f = Fem.from_problem(p)
    print(f"[amg tiles] {kind} {nx}x{ny}", flush=True)
    for _ in range(2):   # (the second with the first one's polling hint)
        info = f.solve(SOLVE_MIXED, tol=1e-8, max_iter=500,
                       opts=solve_opts(MIXED_AMG_FCG, true_residual=True))
        res = f.true_residual()
        print(info["iters"], mirror, res)
        assert info["status"] == 0 and info["iters"] <= mirror + 3, info
        assert res <= 1.001e-8
    f.destroy()
