"""The coarsest level's inverse entry by entry (k_dense_sweep, k_dense_residual,
k_dense_refine).

A system of at most 200 unknowns is preconditioned by that inverse alone, and the
first outer iteration from zero with the unit load e_j gives alpha C^-1 e_j: column
j as it is stored, in FP32, times a scalar.  Each column, scaled to length one,
lies within 2^-23 of the exact inverse's (2^-24 for the rounding of its entries,
the rest for what is left of the inverse's own error), also for elements of 1e-9
of the others' stiffness at condition numbers of 1e11 and 1e12, where an inverse
in FP64 alone is off by 1e-6.  The sizes take 1, 2, 4, 6 and 7 blocks of 32.  The
exact inverse: Gauss-Jordan in long double and two steps of Newton's iteration with
residuals in doubled long double."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LD = np.longdouble


def _split(a):
    t = a * LD(2 ** 32 + 1)
    hi = t - (t - a)
    return hi, a - hi


def _residual(a, x):
    """I - a x by compensated dot products (Dot2) in long double"""
    s, c = np.eye(len(a), dtype=LD), np.zeros_like(a)
    ah, al = _split(-a)
    xh, xl = _split(x)
    for p in range(len(a)):
        col, row = -a[:, p, None], x[None, p]
        h = col * row
        e = ((ah[:, p, None] * xh[None, p] - h) + ah[:, p, None] * xl[None, p]
             + al[:, p, None] * xh[None, p]) + al[:, p, None] * xl[None, p]
        t = s + h
        z = t - s
        c += ((s - (t - z)) + (h - z)) + e
        s = t
    return s + c


def _inverse(a):
    a = a.astype(LD)
    x = a.copy()
    for k in range(len(a)):
        d = 1 / x[k, k]
        f, r = x[:, k] * d, x[k].copy()
        f[k] = r[k] = 0
        x -= np.outer(f, r)
        x[k] = r * d
        x[:, k] = -f
        x[k, k] = d
    for _ in range(2):
        step = x @ _residual(a, x)
        x = x + step
    assert np.abs(step).max() < 1e-15 * np.abs(x).max()   # (the second one)
    return x


def _problem(nx, ny, soft, seed):
    from nbots_amd import synth
    p = synth.cantilever_traction(nx, ny)
    g = np.random.default_rng(seed)
    return dataclasses.replace(
        p, elem_E=np.where(g.random(p.N_elem) < 0.5, 1.0, soft), dv=synth._bc([], [], []),
        ns=synth._bc([], [], []), vtx=np.arange(p.N_nod, dtype=np.uint32))


@pytest.mark.parametrize("nx,ny,soft,seed", [(1, 1, 0.5, 0), (7, 3, 0.5, 0), (7, 3, 1e-9, 0),
                                             (9, 4, 1e-9, 1), (15, 5, 1e-9, 0), (11, 7, 1e-9, 0),
                                             (9, 9, 0.5, 0)])
def test_columns_of_the_inverse(nx, ny, soft, seed):
    from nbots_amd import synth
    from nbots_amd.fem import Fem, MIXED_AMG_FCG, SOLVE_MIXED, solve_opts
    p = _problem(nx, ny, soft, seed)
    print(f"[amg inverse] {nx}x{ny} {soft}: {p.N}", flush=True)
    f = Fem(p.nod, p.conn)
    x, worst = None, 0.0
    for j in range(p.N):
        q = dataclasses.replace(p, nv=synth._bc([j // 2], [1 - j % 2, j % 2],
                                                [1.0 - j % 2, 1.0 * (j % 2)]))
        f.assemble(p.E, p.nu, p.thickness, p.elem_E)
        f.set_bconditions(q)
        if x is None:
            rp, col, val, _ = f.system()
            a = np.zeros((p.N, p.N))
            a[np.repeat(np.arange(p.N), np.diff(rp.astype(np.int64))), col] = val
            x = _inverse(0.5 * (a + a.T))
        F = f.load_vector()
        if not F.any():      # a clamped unknown
            continue
        assert F[j] == 1.0 and np.count_nonzero(F) == 1
        info = f.solve(SOLVE_MIXED, tol=1e-30, max_iter=1, opts=solve_opts(MIXED_AMG_FCG))
        assert info["iters"] == 1 and info["layout"] & 18 == 16
        u = f.displacement()
        want = (x[:, j] / np.sqrt((x[:, j] ** 2).sum())).astype(np.float64)
        u *= np.sign(u @ want) / np.linalg.norm(u)
        worst = max(worst, np.linalg.norm(u - want))
    f.destroy()
    print(worst)
    assert 0.0 < worst <= 2.0 ** -23
