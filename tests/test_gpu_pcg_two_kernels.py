"""The Jacobi-PCG with two kernels per iteration against the oracle, where its
loads and its dispatch can go wrong: sizes around a workgroup, rows of more
blocks than are loaded ahead, matrices that are not symmetric (full rows),
scalar rows that are short, empty of neighbours, or longer than a tile, one
and three unknowns per node, plain CG, and both sides of the size limits.

Bars, those of the other PCG tests (dot products are summed in another order):
cut at 7 iterations the same status and count, tol_reached within 1e-9
relative and x within rel-L2 1e-11; converged the count within 2, x within
1e-10."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cut(A, rp, col, val, b, plain=False, n=7):
    import oracle
    ref = (oracle.cg if plain else oracle.pcg)(rp, col, val, b, max_iter=n, tol=1e-30)
    x, st, it, tr = (A.solve_cg if plain else A.solve_cg_jacobi)(b, max_iter=n, tol=1e-30)
    assert (st, it) == (ref[3], ref[1]) == (1, n)
    assert abs(tr - ref[2]) <= 1e-9 * ref[2]
    assert np.linalg.norm(x - ref[0]) <= 1e-11 * np.linalg.norm(ref[0])


def _converged(A, rp, col, val, b, plain=False):
    import oracle
    tol = 1e-10 * np.linalg.norm(b)
    ref = (oracle.cg if plain else oracle.pcg)(rp, col, val, b, tol=tol, max_iter=20 * b.size)
    x, st, it, tr = (A.solve_cg if plain else A.solve_cg_jacobi)(b, tol=tol, max_iter=20 * b.size)
    assert st == ref[3] == 0 and abs(it - ref[1]) <= 2 and tr <= tol
    assert np.linalg.norm(x - ref[0]) <= 1e-10 * np.linalg.norm(ref[0])


def _fan(spokes):
    """One node with `spokes` neighbours, clamped on part of the rim."""
    from nbots_amd import synth
    t = 2 * np.pi * np.arange(spokes) / spokes
    nod = np.concatenate([[0.0, 0.0], np.stack([np.cos(t), np.sin(t)], 1).reshape(-1)])
    i = np.arange(spokes)
    conn = np.stack([0 * i, 1 + i, 1 + (i + 1) % spokes], 1).astype(np.uint32).reshape(-1)
    z = synth._bc([], [], [])
    return synth.Problem(0, 0, nod, conn, np.arange(1 + spokes, dtype=np.uint32),
                         np.array([0, 3], np.uint32), np.array([1, 2, 3], np.uint32),
                         ds=synth._bc([0], [1, 1], [0.0, 0.0]),
                         nv=synth._bc([0], [1, 1], [0.3, -1.0]), dv=z, ns=z)


def _system(p):
    import oracle
    rp, col = oracle.pattern(p.N_nod, p.conn)
    val, F, _ = oracle.assemble(p, rp, col)
    oracle.set_bconditions(p, rp, col, val, F)
    return rp, col, val, F


@pytest.mark.parametrize("mesh", ["1x1", "15x15", "16x14", "31x7", "63x31", "fan9", "fan40"])
def test_node_matrices(mesh):
    import nbots_amd as nb
    from nbots_amd import synth
    p = (_fan(int(mesh[3:])) if mesh.startswith("fan")
         else synth.cantilever_traction(*(int(a) for a in mesh.split("x"))))
    rp, col, val, F = _system(p)
    A = nb.Sparse.from_csr(rp, col, val, vars_per_node=2)
    assert A.is_blocked() == 1
    _converged(A, rp, col, val, F)
    if p.N > 64:
        _cut(A, rp, col, val, F)
        _cut(A, rp, col, val, F, plain=True)
        # full rows: one entry off symmetry
        v2 = val.copy()
        row = np.repeat(np.arange(p.N), np.diff(rp.astype(np.int64)))
        v2[np.argmax(np.where(row < col, np.abs(val), 0.0))] *= 1.0 + 1e-6
        A.import_values(v2)
        x, info = A.solve(F, mode=0, tol=1e-30, max_iter=7)
        assert info["layout"] == 0
        _cut(A, rp, col, v2, F)
    A.destroy()


def _laplacian(adj, vpn, rng):
    """CSR and handle of a weighted graph Laplacian plus a positive diagonal,
    vpn unknowns per node coupled through random symmetric blocks."""
    import nbots_amd as nb
    A = nb.Sparse.from_graph([a.size for a in adj], adj, vpn)
    rp, col, _ = A.export()
    row = np.repeat(np.arange(rp.size - 1), np.diff(rp.astype(np.int64)))
    c = col.astype(np.int64)
    h = (np.minimum(row, c) * 2654435761 + np.maximum(row, c) * 40503) % 1000003
    val = -(0.1 + h / 1000003.0)
    val[row == c] = 0.0
    dg = np.bincount(row, -val, minlength=rp.size - 1) + rng.uniform(0.01, 0.1, rp.size - 1)
    val[row == c] = dg
    A.import_values(val)
    return A, rp, col, val


def _grid_adj(nx, ny):
    i = np.arange(nx * ny).reshape(ny, nx)
    e = np.concatenate([np.stack([i[:, :-1].ravel(), i[:, 1:].ravel()], 1),
                        np.stack([i[:-1].ravel(), i[1:].ravel()], 1)])
    e = np.concatenate([e, e[:, ::-1]])
    key = np.unique(e[:, 0] * nx * ny + e[:, 1])
    deg = np.bincount(key // (nx * ny), minlength=nx * ny)
    return np.split((key % (nx * ny)).astype(np.uint32), np.cumsum(deg)[:-1])


@pytest.mark.parametrize("case", ["single", "no_neighbours_300", "grid_16x16", "grid_257x3",
                                  "star_9000", "grid_40x31x3"])
def test_scalar_matrices(case):
    rng = np.random.default_rng(3)
    vpn = 1
    if case == "single":
        adj = [np.zeros(0, np.uint32)]
    elif case == "no_neighbours_300":   # rows of one entry
        adj = [np.zeros(0, np.uint32)] * 300
    elif case == "star_9000":           # one row over two tiles long, the rest of two entries
        adj = [np.arange(1, 9000, dtype=np.uint32)] + [np.zeros(1, np.uint32)] * 8999
    else:
        d = [int(a) for a in case[5:].split("x")]
        adj, vpn = _grid_adj(d[0], d[1]), (d + [1])[2]
    A, rp, col, val = _laplacian(adj, vpn, rng)
    assert A.is_blocked() == 0
    b = rng.standard_normal(rp.size - 1)
    if rp.size - 1 == col.size:   # diagonal: exact after one step, 0/0 after the next
        _cut(A, rp, col, val, b, n=1)
        return
    _converged(A, rp, col, val, b)
    if case.startswith("grid"):
        _cut(A, rp, col, val, b)
        _cut(A, rp, col, val, b, plain=True)
    A.destroy()


@pytest.mark.parametrize("n", [(362, 362), (363, 362), (512, 512), (513, 512)])
def test_scalar_limits(n):
    """131,044 and 131,406 rows (the tile sizes), 262,144 and 262,656 (two
    kernels and five)."""
    rng = np.random.default_rng(4)
    A, rp, col, val = _laplacian(_grid_adj(*n), 1, rng)
    _cut(A, rp, col, val, rng.standard_normal(rp.size - 1))
    A.destroy()


@pytest.mark.parametrize("n", [(361, 361), (362, 361), (442, 442), (443, 443)])
def test_node_limits(n):
    """131,044 and 131,406 nodes, 196,249 (two kernels) and 197,136 (five),
    through the device system in reference mode."""
    import oracle
    from nbots_amd import synth
    from nbots_amd.fem import Fem, SOLVE_REFERENCE
    p = synth.cantilever_traction(*n)
    rp, col, val, F = _system(p)
    ref = oracle.pcg(rp, col, val, F, max_iter=7, tol=1e-30)
    f = Fem.from_problem(p)
    i = f.solve(SOLVE_REFERENCE, tol=1e-30, max_iter=7)
    assert (i["status"], i["iters"], i["layout"]) == (1, 7, 1)
    assert abs(i["tol_reached"] - ref[2]) <= 1e-9 * ref[2]
    u = f.displacement()
    assert np.linalg.norm(u - ref[0]) <= 1e-11 * np.linalg.norm(ref[0])
    f.destroy()
