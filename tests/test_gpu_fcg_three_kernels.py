"""The flexible CG with three kernels around its preconditioner, cut after a
few outer iterations: the residual norm it carries along (through alpha, beta,
the directions and both state slots) against the one of its iterate, computed
afresh.  Sizes of one node row to one workgroup and over, both sides of the
limit (262,144 nodes; seven kernels above it), symmetric and full rows, each
preconditioner.  Three steps drift by a few roundings of ||K|| ||x|| / ||r||,
under 1e-9 here: bar 1e-8 relative.  With no step allowed and with the exact
solution as the start the first kernel alone decides."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _variants():
    from nbots_amd.fem import MIXED_AMG_FCG, MIXED_CHEB_FCG, solve_opts
    return {"cheb16": solve_opts(MIXED_CHEB_FCG, cheb_degree=6),
            "cheb32": solve_opts(MIXED_CHEB_FCG, cheb_degree=6, precond_bits=32),
            "amg": solve_opts(MIXED_AMG_FCG)}


@pytest.mark.parametrize("steps", [1, 2, 3])
@pytest.mark.parametrize("variant", ["cheb16", "cheb32", "amg"])
@pytest.mark.parametrize("n", [(3, 2), (31, 7), (32, 8), (140, 70)])
def test_carried_residual(n, variant, steps):
    from nbots_amd import synth
    from nbots_amd.fem import Fem, SOLVE_MIXED
    f = Fem.from_problem(synth.cantilever_traction(*n))
    o = _variants()[variant]
    i = f.solve(SOLVE_MIXED, tol=1e-14, max_iter=steps, opts=o)
    r = f.true_residual()
    if r < 1e-9:   # 3x2 with the dense coarsest solve: at the rounding of K x itself
        assert n == (3, 2) and variant == "amg"
        return
    assert (i["status"], i["iters"]) == (1, steps)
    assert abs(i["rel_res"] - r) <= 1e-8 * r, (i["rel_res"], r)
    f.destroy()


@pytest.mark.parametrize("n", [(511, 511), (512, 511)])
def test_carried_residual_at_the_limit(n):
    from nbots_amd import synth
    from nbots_amd.fem import Fem, SOLVE_MIXED
    f = Fem.from_problem(synth.cantilever_traction(*n))
    i = f.solve(SOLVE_MIXED, tol=1e-14, max_iter=3, opts=_variants()["cheb16"])
    r = f.true_residual()
    assert (i["status"], i["iters"]) == (1, 3) and abs(i["rel_res"] - r) <= 1e-8 * r
    f.destroy()


def test_full_rows_and_ends():
    import nbots_amd as nb
    import oracle
    from nbots_amd import synth
    from nbots_amd.fem import Fem, SOLVE_MIXED
    p = synth.cantilever_traction(31, 8)
    f = Fem.from_problem(p)
    rp, col, val, F = f.system()
    o = _variants()["cheb16"]
    # no step allowed: the iterate stays the start
    i = f.solve(SOLVE_MIXED, tol=1e-8, max_iter=0, opts=o)
    assert (i["status"], i["iters"], i["rel_res"]) == (1, 0, 1.0) and not f.displacement().any()
    # the start already meets the tolerance
    u = oracle.pcg(rp, col, val, F, tol=1e-13 * np.linalg.norm(F), max_iter=20 * p.N)[0]
    i = f.solve(SOLVE_MIXED, tol=1e-8, u0=u, opts=o)
    assert (i["status"], i["iters"]) == (0, 0) and np.array_equal(f.displacement(), u)
    f.destroy()
    row = np.repeat(np.arange(p.N), np.diff(rp.astype(np.int64)))
    val[np.argmax(np.where(row < col, np.abs(val), 0.0))] *= 1.0 + 1e-6
    A = nb.Sparse.from_csr(rp, col, val, vars_per_node=2)
    x, i = A.solve(F, mode=SOLVE_MIXED, tol=1e-14, max_iter=3, opts=o)
    r = np.linalg.norm(F - oracle.spmv(rp, col, val, x)) / np.linalg.norm(F)
    assert (i["status"], i["iters"], i["layout"] & 1) == (1, 3, 0)
    assert abs(i["rel_res"] - r) <= 1e-8 * r
    A.destroy()
