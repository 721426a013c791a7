"""Performance cases of the FEM solve path: what a program that uses this
package has it do, each through the public entry points (the drop-in nb_* API,
the device-resident nbx_fem_* system and the nbx_simp_* loop).

listed() gives the fixed cases, draw(rng) one more of the same ranges,
prepare(case, seed) the inputs and handles a program has in hand, run(state)
one pass, work(case) the bytes and operations a pass cannot do without, and
exact(case, seed) the results in 64 bits from a plain torch model (element
matrices and a block-tridiagonal direct solve) that shares no code with the
package.

Sizes are elements per side (nx x ny squares, each cut into two triangles), as
in the package's synthetic problems: 64x32 is the smallest cantilever of its
tests, 1024x512 and 2048x1024 the benchmark's.
"""
import ctypes as C
import functools
import math

import numpy as np
import torch

from nbots_amd import Sparse, load, synth
from nbots_amd.fem import (MIXED_AMG_FCG, SOLVE_FP64, SOLVE_MIXED, Fem, Simp,
                           compute_2D_solid_mechanics, solve_opts)

RTOL = 1e-8          # the package's default relative tolerance
GRAD_RTOL = 1e-10    # its default for adjoint solves, taken where strains and
                     # gradients follow from a reduced-precision solve
AMG_MAX_ITER = 5000


# ---- what is measured -------------------------------------------------------
def listed():
    return [
        # A C or Python caller of the reference's driver on its own small
        # test size: objects in, displacement, strain and stress out.
        # Latency and launches count.
        dict(name="driver_64x32", kind="driver", nx=64, ny=32),
        # Jacobi-PCG on a scalar CSR already on the GPU, for callers that
        # bring their own matrix and may not allocate (41,004 rows).
        dict(name="device_csr_200x101", kind="device_csr", nx=200, ny=101),
        # The drop-in product nb_sparse_multiply_vector on host vectors, as
        # an eigenvalue or time-stepping loop of the reference calls it.
        dict(name="matvec_256x128", kind="matvec", nx=256, ny=128),
        # FP64 Jacobi-PCG on a resident system, the reference's algorithm: a
        # medium mesh, and the 1.05M-DOF cantilever.
        dict(name="fp64_256x128", kind="fp64", nx=256, ny=128),
        dict(name="fp64_1024x512", kind="fp64", nx=1024, ny=512),
        # The default solve (Chebyshev-preconditioned, mixed precision) at an
        # odd, ragged size.
        dict(name="mixed_501x247", kind="mixed", nx=501, ny=247),
        # Multigrid-preconditioned solves on a resident system (one load
        # after another on one matrix): a small mesh and the largest
        # benchmark size, 4.2M DOF.
        dict(name="amg_150x75", kind="amg", nx=150, ny=75),
        dict(name="amg_2048x1024", kind="amg", nx=2048, ny=1024),
        # A whole analysis from mesh arrays to strain and stress, once per
        # mesh: pattern, assembly, conditions, default solve, results.
        dict(name="analysis_300x150", kind="analysis", nx=300, ny=150),
        # One evaluation of an objective and its gradients for an outside
        # optimiser (MMA, L-BFGS, an autograd function): new moduli,
        # conditions, state solve, compliance gradient, adjoint solve.
        dict(name="gradient_256x128", kind="gradient", nx=256, ny=128),
        # Topology optimisation from a given design: the filter and the first
        # design iterations, at a small and at a large size.
        dict(name="simp_96x48", kind="simp", nx=96, ny=48, iters=8),
        dict(name="simp_512x256", kind="simp", nx=512, ny=256, iters=8),
    ]


#: kind -> smallest and largest nx of a drawn case
RANGES = dict(driver=(16, 128), device_csr=(24, 320), matvec=(24, 320), fp64=(24, 800),
              mixed=(24, 800), amg=(24, 1400), analysis=(24, 500), gradient=(24, 400),
              simp=(32, 400))


def draw(rng):
    kind = rng.choice(sorted(RANGES))
    lo, hi = RANGES[kind]
    nx = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    ny = max(8, int(round(nx * rng.uniform(0.35, 0.6))))
    case = dict(kind=kind, nx=nx, ny=ny)
    if kind == "simp":
        case["iters"] = rng.randint(4, 8)
    return case


# ---- inputs -----------------------------------------------------------------
@functools.lru_cache(maxsize=4)
def _grid(nx, ny):
    return synth.grid(nx, ny)


def _traction(nx, ny, seed, jitter=0.0):
    """Cantilever with lognormal moduli, clamped left, sheared on the right."""
    nod, conn, vtx, sp, sn = _grid(nx, ny) if jitter == 0.0 else synth.grid(nx, ny, 1.0, jitter,
                                                                            seed)
    rng = np.random.default_rng(seed)
    z = np.zeros(0, np.uint32), np.zeros(0, np.uint8), np.zeros(0)
    return synth.Problem(nx, ny, nod, conn, vtx, sp, sn,
                         elem_E=np.exp(rng.standard_normal(conn.size // 3)), dv=z, nv=z,
                         ds=(np.array([3], np.uint32), np.array([1, 1], np.uint8), np.zeros(2)),
                         ns=(np.array([1], np.uint32), np.array([0, 1], np.uint8),
                             np.array([0.0, -float(ny)])))


def _problem(case, seed):
    kind, nx, ny = case["kind"], case["nx"], case["ny"]
    if kind == "driver":
        return synth.cantilever_point(nx, ny, jitter=0.1, seed=seed)
    if kind == "analysis":
        return _traction(nx, ny, seed, jitter=0.1)
    if kind in ("gradient", "simp"):
        rng = np.random.default_rng(seed)
        lo, hi = (0.3, 1.0) if kind == "gradient" else (0.4, 0.6)
        return synth.mbb(nx, ny, rho=rng.uniform(lo, hi, 2 * nx * ny))
    return _traction(nx, ny, seed)


def _objective(case, seed):
    """dL/du of L = sum of weighted vertical displacements of the top edge."""
    nx, ny = case["nx"], case["ny"]
    g = np.zeros(2 * (nx + 1) * (ny + 1))
    top = ny * (nx + 1) + np.arange(nx + 1)
    g[2 * top + 1] = np.random.default_rng(seed + 1).uniform(0.5, 1.5, nx + 1) / (nx + 1)
    return g


def _vector(case, seed):
    n = 2 * (case["nx"] + 1) * (case["ny"] + 1)
    return np.random.default_rng(seed + 2).standard_normal(n)


@functools.lru_cache(maxsize=2)
def _adjacency(nx, ny):
    """The mesh's node graph as the reference's per-node neighbour lists."""
    conn = _grid(nx, ny)[1].reshape(-1, 3).astype(np.int64)
    e = np.concatenate([conn[:, [0, 1]], conn[:, [1, 2]], conn[:, [2, 0]]])
    e = np.concatenate([e, e[:, ::-1]])
    n = (nx + 1) * (ny + 1)
    key = np.unique(e[:, 0] * n + e[:, 1])
    deg = np.bincount(key // n, minlength=n)
    return deg, np.split((key % n).astype(np.uint32), np.cumsum(deg)[:-1])


def _dev(a, dtype):
    return torch.from_numpy(a).to("cuda", dtype)


def prepare(case, seed):
    kind = case["kind"]
    p = _problem(case, seed)
    s = dict(kind=kind, p=p)
    if kind in ("driver", "analysis"):
        return s
    s["fem"] = f = Fem.from_problem(p)
    if kind == "device_csr":
        rp, col, val, F = f.system()
        s["csr"] = [_dev(rp.view(np.int32), torch.int32), _dev(col.view(np.int32), torch.int32),
                    _dev(val, torch.float64)]
        s["b"] = _dev(F, torch.float64)
        s["x"] = torch.zeros_like(s["b"])
        s["tol"] = RTOL * float(np.linalg.norm(F))
        del s["fem"]
    elif kind == "matvec":
        _, _, val, _ = f.system()
        s["A"] = Sparse.from_graph(*_adjacency(case["nx"], case["ny"]), vars_per_node=2)
        s["A"].import_values(val)
        s["x"] = _vector(case, seed)
        del s["fem"]
    elif kind == "amg":
        s["opts"] = solve_opts(MIXED_AMG_FCG)
    elif kind == "gradient":
        s["opts"] = solve_opts(MIXED_AMG_FCG)
        s["dLdu"] = _objective(case, seed)
    elif kind == "simp":
        s["iters"] = case["iters"]
    return s


# ---- one pass ---------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind == "driver":
        _, u, strain, stress = compute_2D_solid_mechanics(s["p"])
        return u, strain, stress
    if kind == "device_csr":
        b, x = s["b"], s["x"]
        x.zero_()
        it, tr = C.c_uint32(), C.c_double()
        rc = load().nbx_sparse_solve_CG_precond_Jacobi_noalloc(
            b.numel(), *(t.data_ptr() for t in s["csr"]), b.data_ptr(), x.data_ptr(), b.numel(),
            s["tol"], C.byref(it), C.byref(tr), None)
        if rc != 0:
            raise RuntimeError("the solve did not converge")
        return x
    if kind == "matvec":
        return s["A"].matvec(s["x"])
    if kind == "analysis":
        p = s["p"]
        f = Fem.from_problem(p)
        f.solve(SOLVE_MIXED, tol=GRAD_RTOL)
        u = f.displacement()
        strain, stress = f.strain_stress()
        f.destroy()
        return u, strain, stress
    f = s["fem"]
    if kind == "fp64":
        f.solve(SOLVE_FP64, tol=RTOL)
        return f.displacement()
    if kind == "mixed":
        f.solve(SOLVE_MIXED, tol=GRAD_RTOL)
        return f.displacement()
    if kind == "amg":
        f.solve(SOLVE_MIXED, tol=RTOL, max_iter=AMG_MAX_ITER, opts=s["opts"])
        return f.displacement()
    p = s["p"]
    if kind == "gradient":
        f.assemble(p.E, p.nu, p.thickness, p.elem_E)
        f.set_bconditions(p)
        f.solve(SOLVE_MIXED, tol=GRAD_RTOL, max_iter=AMG_MAX_ITER, opts=s["opts"])
        comp, dc, _ = f.compliance(p.rho)
        lam, _ = f.adjoint(s["dLdu"], mode=SOLVE_MIXED, rtol=GRAD_RTOL)
        return comp, dc, f.elem_cross(lam)
    o = Simp(f, x0=p.rho)
    hist = [o.iterate()[0] for _ in range(s["iters"])]
    x, xphys, dc, _ = o.state()
    o.destroy()
    return np.array(hist), x, xphys, dc


# ---- what a pass cannot do without ------------------------------------------
def work(case):
    """Inputs read once, outputs written once; a solve counts one pass over
    its matrix (12 B per entry, the index and the FP64 value) and vectors."""
    kind, nx, ny = case["kind"], case["nx"], case["ny"]
    n_nod, ne = (nx + 1) * (ny + 1), 2 * nx * ny
    nnz = 4.0 * (n_nod + 2 * (nx * (ny + 1) + ny * (nx + 1) + nx * ny))
    n = 2.0 * n_nod
    mesh, matrix, vec = 16.0 * n_nod + 12.0 * ne, 12.0 * nnz, 8.0 * n
    elem = 8.0 * ne
    if kind in ("driver", "analysis"):
        return dict(bytes=mesh + elem + matrix + vec + 6 * elem, flops=4 * nnz + 150.0 * ne)
    if kind in ("device_csr", "matvec", "fp64", "mixed", "amg"):
        return dict(bytes=matrix + 2 * vec, flops=2 * nnz)
    if kind == "gradient":
        return dict(bytes=mesh + elem + matrix + 3 * vec + 4 * elem, flops=4 * nnz + 150.0 * ne)
    # each iteration needs the design, the filter (about 14 entries of 12 B per
    # element at radius 1.5) twice, K once and the displacement
    it = case["iters"]
    return dict(bytes=mesh + it * (matrix + 2 * vec + 2 * 14 * 12.0 * ne + 6 * elem),
                flops=it * (2 * nnz + 2 * 28.0 * ne + 150.0 * ne))


# ---- the results in 64 bits -------------------------------------------------
def _plate(p):
    """Element matrices [ne, 6, 6] at unit modulus, dof lists, B and area."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    xy = torch.from_numpy(p.nod.reshape(-1, 2)).to(dev)
    conn = torch.from_numpy(p.conn.reshape(-1, 3).astype(np.int64)).to(dev)
    q = xy[conn]
    x, y = q[..., 0], q[..., 1]
    j, k = [1, 2, 0], [2, 0, 1]
    by, bx = y[:, j] - y[:, k], x[:, k] - x[:, j]
    area = 0.5 * ((x[:, 1] - x[:, 0]) * (y[:, 2] - y[:, 0])
                  - (x[:, 2] - x[:, 0]) * (y[:, 1] - y[:, 0]))
    B = torch.zeros(conn.shape[0], 3, 6, dtype=torch.float64, device=dev)
    B[:, 0, 0::2] = by
    B[:, 1, 1::2] = bx
    B[:, 2, 0::2] = bx
    B[:, 2, 1::2] = by
    B = B / (2 * area)[:, None, None]
    d0 = 1.0 / (1.0 - p.nu ** 2)
    D = torch.tensor([[d0, p.nu * d0, 0], [p.nu * d0, d0, 0], [0, 0, 0.5 / (1 + p.nu)]],
                     dtype=torch.float64, device=dev)
    DB = (D[None, :, :, None] * B[:, None, :, :]).sum(2)
    K0 = (B[:, :, :, None] * DB[:, :, None, :]).sum(1) * (area * p.thickness)[:, None, None]
    dof = torch.stack([2 * conn, 2 * conn + 1], -1).reshape(-1, 6)
    return K0, dof, B, D


def _loads(p):
    """(F before elimination, constrained dofs), zero Dirichlet values."""
    F, fixed = np.zeros(p.N), []
    ids, mask, val = p.nv
    for c, i in enumerate(ids):
        for d in range(2):
            F[2 * p.vtx[i] + d] += val[2 * c + d] if mask[2 * c + d] else 0.0
    ids, mask, val = p.ns
    for c, i in enumerate(ids):
        nodes = p.sgm_nodes[p.sgm_ptr[i]:p.sgm_ptr[i + 1]].astype(np.int64)
        q = p.nod.reshape(-1, 2)[nodes]
        share = np.linalg.norm(np.diff(q, axis=0), axis=1)
        share /= share.sum()
        for d in range(2):
            if mask[2 * c + d]:
                np.add.at(F, 2 * nodes[:-1] + d, 0.5 * share * val[2 * c + d])
                np.add.at(F, 2 * nodes[1:] + d, 0.5 * share * val[2 * c + d])
    for (ids, mask, _), nodes_of in ((p.ds, lambda i: p.sgm_nodes[p.sgm_ptr[i]:p.sgm_ptr[i + 1]]),
                                     (p.dv, lambda i: p.vtx[i:i + 1])):
        for c, i in enumerate(ids):
            fixed += [2 * nodes_of(i).astype(np.int64) + d for d in range(2) if mask[2 * c + d]]
    fixed = np.unique(np.concatenate(fixed))
    F[fixed] = 0.0
    return F, fixed


class _Direct:
    """Block-tridiagonal Cholesky of the plate, one block per grid column."""

    def __init__(self, p):
        self.K0, self.dof, self.B, self.D = _plate(p)
        dev = self.K0.device
        E = np.full(p.N_elem, p.E) if p.elem_E is None else p.elem_E
        self.E = torch.from_numpy(E).to(dev)
        self.F, fixed = _loads(p)
        self.nb, self.m = p.nx + 1, 2 * (p.ny + 1)
        node = torch.arange(p.N_nod, device=dev)
        col, row = node % self.nb, node // self.nb
        place = torch.stack([2 * row, 2 * row + 1], -1).reshape(-1)      # within the block
        block = col.repeat_interleave(2)
        self.perm = torch.empty(p.N, dtype=torch.int64, device=dev)
        self.perm[block * self.m + place] = torch.arange(p.N, device=dev)
        free = torch.ones(p.N, dtype=torch.bool, device=dev)
        free[torch.from_numpy(fixed).to(dev)] = False
        self.free = free
        Ke = self.K0 * self.E[:, None, None]
        keep = free[self.dof]
        Ke = Ke * keep[:, :, None] * keep[:, None, :]
        r = self.dof[:, :, None].expand(-1, 6, 6).reshape(-1)
        c = self.dof[:, None, :].expand(-1, 6, 6).reshape(-1)
        v, m = Ke.reshape(-1), self.m
        self.Dg = torch.zeros(self.nb * m * m, dtype=torch.float64, device=dev)
        self.Up = torch.zeros(self.nb * m * m, dtype=torch.float64, device=dev)
        at = block[r] * m * m + place[r] * m + place[c]
        for out, step in ((self.Dg, 0), (self.Up, 1)):
            t = block[c] - block[r] == step
            out.index_add_(0, at[t], v[t])
        fx = torch.from_numpy(fixed).to(dev)
        self.Dg[block[fx] * m * m + place[fx] * (m + 1)] = 1.0
        self.Dg, self.Up = self.Dg.view(-1, m, m), self.Up.view(-1, m, m)
        self.L, self.V = [], []
        S = self.Dg[0]
        for i in range(self.nb):
            L = torch.linalg.cholesky(S)
            self.L.append(L)
            if i + 1 < self.nb:
                V = torch.linalg.solve_triangular(L, self.Up[i], upper=False)
                self.V.append(V)
                S = self.Dg[i + 1] - V.t().contiguous() @ V

    def _times(self, x):
        y = torch.zeros_like(x)
        for i in range(self.nb):
            y[i] += self.Dg[i] @ x[i]
            if i + 1 < self.nb:
                y[i] += self.Up[i] @ x[i + 1]
                y[i + 1] += self.Up[i].t() @ x[i]
        return y

    def _solve(self, b):
        y = torch.empty_like(b)
        for i in range(self.nb):
            t = b[i] if i == 0 else b[i] - self.V[i - 1].t() @ y[i - 1]
            y[i] = torch.linalg.solve_triangular(self.L[i], t[:, None], upper=False)[:, 0]
        for i in reversed(range(self.nb)):
            t = y[i] if i + 1 == self.nb else y[i] - self.V[i] @ y[i + 1]
            y[i] = torch.linalg.solve_triangular(self.L[i].t(), t[:, None], upper=True)[:, 0]
        return y

    def solve(self, rhs):
        b = torch.as_tensor(rhs, device=self.free.device) * self.free
        bb = b[self.perm].view(self.nb, self.m)
        x = self._solve(bb)
        for _ in range(2):
            x = x + self._solve(bb - self._times(x))
        u = torch.empty_like(b)
        u[self.perm] = x.reshape(-1)
        return u

    def times(self, x):
        """K x after the elimination."""
        xx = torch.as_tensor(x, device=self.free.device)[self.perm].view(self.nb, self.m)
        y = torch.empty(xx.numel(), dtype=torch.float64, device=xx.device)
        y[self.perm] = self._times(xx).reshape(-1)
        return y

    def strain_stress(self, u):
        e = (self.B * u[self.dof][:, None, :]).sum(2)
        s = (self.D[None] * e[:, None, :]).sum(2) * self.E[:, None]
        return e.reshape(-1), s.reshape(-1)

    def cross(self, a, b):
        t = (self.K0 * b[self.dof][:, None, :]).sum(2)
        return (a[self.dof] * t).sum(1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "simp" or case["nx"] * case["ny"] > 600_000:   # too long for a direct solve
        return None
    p = _problem(case, seed)
    K = _Direct(p)

    def out(t):
        return t.cpu() if kind == "device_csr" else t.cpu().numpy()

    if kind == "matvec":
        return out(K.times(_vector(case, seed)))
    u = K.solve(K.F)
    if kind in ("driver", "analysis"):
        return tuple(out(t) for t in (u, *K.strain_stress(u)))
    if kind == "gradient":
        ce = K.cross(u, u)
        rho = torch.from_numpy(p.rho).to(u.device)
        dc = -3.0 * rho ** 2 * (1.0 - 1e-9) * ce
        lam = K.solve(_objective(case, seed))
        return float((K.E * ce).sum()), out(dc), out(K.cross(lam, u))
    return out(u)
