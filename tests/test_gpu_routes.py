"""Which kernels a solve runs: the rules that choose between several steps per
launch and one leave the results and most times alike, so the tests of those
kernels would pass without them.  A child process records the kernels of two
outer iterations on the meshes of those tests (torch's profiler sees every kernel
of the process), and each mesh has to have run the form it stands for.

Also the largest tiles' rule (three rings beyond 1,024 * 528 nodes) bit for bit
against the sparse API's single steps, on both sides."""
import json
import os
import re
import subprocess
import sys

import pytest

import test_gpu_cheb_tiles as cheb
from conftest import ROOT

pytestmark = pytest.mark.gpu

CHILD = r'''
import json, re, sys
sys.path[:0] = [".", "tests"]
import torch
from torch.profiler import ProfilerActivity, profile
import test_gpu_amg_bottom as amg
import test_gpu_amg_layouts as layouts
import test_gpu_cheb_tiles as cheb
import test_gpu_cheb_tiles_uneven as uneven
from nbots_amd.fem import Fem, MIXED_AMG_FCG, SOLVE_MIXED, solve_opts

torch.zeros(1, device="cuda")


def kernels(p, opts=None):
    f = Fem.from_problem(p)
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        f.solve(SOLVE_MIXED, tol=1e-8, max_iter=2, opts=opts)
        torch.cuda.synchronize()
    f.destroy()
    found = (re.match(r"(?:void )?nbx::(?:\(anonymous namespace\)::)?(k_\w+(?:<[^(]*>)?)\(", e.key)
             for e in prof.key_averages())
    return sorted({m.group(1) for m in found if m})


def mesh(case):
    kind, args = case[0], case[1:]
    if kind == "named":
        return cheb.MESHES[args[0]]()
    if kind == "hub":
        return layouts.hub(*args)
    return {"grid": cheb._grid, "delaunay": amg.delaunay, "point": lambda *n: amg.mesh("grid", *n),
            "graded": uneven._graded}[kind](*args)


o = solve_opts(MIXED_AMG_FCG)
for solver, case in json.loads(sys.argv[1]):
    print("ROUTE", json.dumps([solver, case, kernels(mesh(case), o if solver == "amg" else None)]),
          flush=True)
'''

D6, F6, F12 = (f"k_cheb_tiles<{t}>" for t in ("6, true, double", "6, true, float",
                                              "12, false, float"))
STEP = "k_cheb_step64"
# solver, mesh, kernels that have to run, kernels that must not
CASES = [
    *[("cheb", ("named", m), [D6], [STEP]) for m in
      ("below_a_tile_5x3", "one_tile_15x9", "64x32_jitter", "odd_131x67", "crowded_96x48",
       "shuffled_60x41")],
    *[("cheb", ("named", m), [F12], [STEP]) for m in ("slab_700x3", "beam_mesh", "plate_mesh")],
    *[("cheb", ("grid", *n), [D6], [STEP]) for n in ((362, 181), (363, 181), (442, 220))],
    *[("cheb", ("grid", *n), [F6], [STEP]) for n in ((446, 220), (570, 287), (811, 403),
                                                     (1038, 519), (1039, 519))],
    ("cheb", ("graded", 724, 362), [STEP], ["k_cheb_tiles"]),
    ("amg", ("point", 34, 17), ["k_amg_bottom<512, 14, 2>"], ["k_amg_down", "k_bsm_step"]),
    ("amg", ("point", 54, 27), ["k_amg_bottom<1024, 14, 2>"], ["k_amg_down", "k_bsm_step"]),
    ("amg", ("point", 76, 38), ["k_amg_bottom<1024, 14, 2>"], ["k_amg_down", "k_bsm_step"]),
    ("amg", ("point", 77, 39), ["k_amg_down<512, 14, 2>", "k_amg_up<512, 14, 2>", "k_amg_dense"],
     ["k_amg_bottom", "k_bsm_step"]),
    ("amg", ("point", 96, 48), ["k_amg_down<512, 14, 4>", "k_amg_up<512, 14, 4>", "k_amg_dense"],
     ["k_amg_bottom", "k_bsm_step"]),
    ("amg", ("point", 333, 12), ["k_amg_down<512, 14, 2>", "k_amg_bottom<512, 14, 2>"],
     ["k_bsm_step"]),
    ("amg", ("point", 448, 224), ["k_amg_down<1024, 14, 4>", "k_amg_bottom<512, 14, 2>"],
     ["k_bsm_step"]),
    ("amg", ("delaunay", 40, 20), ["k_amg_bottom<512, 24, 4>"], ["k_amg_down", "k_bsm_step"]),
    ("amg", ("delaunay", 64, 32), ["k_amg_down<512, 24, 4>", "k_amg_dense"],
     ["k_amg_bottom", "k_bsm_step"]),
    ("amg", ("delaunay", 128, 64), ["k_amg_down<512, 24, 4>", "k_amg_bottom<512, 24, 4>"],
     ["k_bsm_step"]),
    # a launch per step on a small level (rows of more than 24 blocks), four
    # lanes a row, and on a large one, one lane
    ("amg", ("hub", 48, 24), ["k_bsm_step<false, 4, 4>", "k_bsm_init<4, 4>", "k_bresidual<4, 4>",
                              "k_amg_dense"], ["k_amg_bottom", "k_amg_down"]),
    ("amg", ("point", 1024, 512), ["k_bsm_step<false, 4, 1>", "k_bresidual<4, 1>",
                                   "k_amg_down<1024, 14, 4>"], []),
]


@pytest.fixture(scope="module")
def routes():
    r = subprocess.run([sys.executable, "-u", "-c", CHILD,
                        json.dumps([c[:2] for c in CASES])], cwd=ROOT, capture_output=True,
                       text=True, timeout=240, env=dict(os.environ))
    got = [json.loads(line[6:]) for line in r.stdout.splitlines() if line.startswith("ROUTE ")]
    assert r.returncode == 0 and len(got) == len(CASES), r.stdout[-2000:] + r.stderr[-2000:]
    return {(solver, tuple(case)): names for solver, case, names in got}


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(a) for a in (c[0], *c[1])))
def test_route(routes, case):
    solver, mesh, run, not_run = case
    names = routes[(solver, mesh)]
    print(names)
    assert all(any(n.startswith(k) for n in names) for k in run)
    assert not any(re.match(k + r"\b", n) for n in names for k in not_run)


@pytest.mark.parametrize("n", [(1038, 519), (1039, 519)])
def test_largest_tiles_equal_single_steps(n):
    """540,280 and 540,800 nodes"""
    cheb.test_tiles_equal_single_steps_at_the_rules_edges(n)
