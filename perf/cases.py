"""Timed workloads of the assembly-and-solve path, through the package's public entry points.

listed()            the workloads, each a dict of plain values with a name
draw(rng)           one more workload from the same ranges (rng: random.Random)
prepare(case, seed) the device system a program holds before the call: mesh, dofs, pattern, cell
                    values, colours, constraints, and the seeded coefficients
run(state)          one pass; returns what the pass computes (K.nzval, f, u, gradients)
work(case)          bytes and flops a pass cannot do without: every input read once, every output
                    written once; assembly flops and one operator application of a solve
exact(case, seed)   the same outputs from plain torch / numpy in 64 bits

Kinds of work
  poisson     one load step -div(k grad u) = s with scalar Q1 elements: assembly, apply!, CG solve
              to 1e-10, u copied to the host; quads with u = 0 on the whole boundary, or hexes with
              u = 0 on two opposite faces; box or distorted meshes; FP64 or mixed solver
  assembly    assembly and apply! alone (the matrix stays on the device for the program's own use)
  elasticity  Q2 hex elasticity: assembly, traction, apply!, with or without the solve
  compliance  one step of a SIMP design loop: plane-strain Q1 cantilever, assembly, point load,
              apply!, CG to 2e-9, J and both adjoint gradients
  batch       many independent Poisson problems assembled, constrained and solved in one call
"""
import ctypes
import functools
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ferrite.jl_amd"))

import ferrite_amd as fa  # noqa: E402
from ferrite_amd import _lib as L  # noqa: E402
from ferrite_amd.autodiff import ComplianceProblem  # noqa: E402
from ferrite_amd.batch import BatchedPoisson, poisson_problem  # noqa: E402

RTOL = 1e-10
NU, EMIN, PENAL = 0.3, 1e-3, 3.0


def listed():
    return [
        # the heat-equation tutorial: the smallest call, all latency and launches
        dict(name="heat-quad-20", kind="poisson", nx=20, ny=20, nz=0, coef=False, distort=False, mode="cg"),
        # the same at the usual size of a 2D study
        dict(name="heat-quad-100", kind="poisson", nx=100, ny=100, nz=0, coef=False, distort=False, mode="cg"),
        # heterogeneous 2D diffusion on an odd grid, mixed-precision solver
        dict(name="diffusion-quad-301x227", kind="poisson", nx=301, ny=227, nz=0, coef=True, distort=False, mode="mixed"),
        # a small unstructured-style 3D mesh: the general operator, FP64
        dict(name="poisson-hex-24x20x17-dist", kind="poisson", nx=24, ny=20, nz=17, coef=True, distort=True, mode="cg"),
        # an ordinary distorted 3D mesh, mixed-precision solver
        dict(name="poisson-hex-47x53x61-dist", kind="poisson", nx=47, ny=53, nz=61, coef=True, distort=True, mode="mixed"),
        # an ordinary box, default FP64 solver
        dict(name="poisson-hex-64", kind="poisson", nx=64, ny=64, nz=64, coef=True, distort=False, mode="cg"),
        # the headline workload of the benchmark
        dict(name="poisson-hex-128-mixed", kind="poisson", nx=128, ny=128, nz=128, coef=True, distort=False, mode="mixed"),
        # a re-assembly inside a program that has its own solver
        dict(name="assembly-hex-96x101x90-dist", kind="assembly", nx=96, ny=101, nz=90, coef=True, distort=True, precision="fp64"),
        # Q2 elasticity assembly, the largest matrix per cell
        dict(name="elasticity-q2-30x28x26", kind="elasticity", nx=30, ny=28, nz=26, precision="fp64", mode="none"),
        # a whole Q2 elasticity step: FP32 matrix-core element products, mixed solver
        dict(name="elasticity-q2-12x10x9-solve", kind="elasticity", nx=12, ny=10, nz=9, precision="mixed", mode="mixed"),
        # one step of the topology-optimisation cantilever with its gradients
        dict(name="compliance-512x256", kind="compliance", nx=512, ny=256),
        # a parameter study: many problems of mixed sizes and dimensions
        dict(name="batch-24", kind="batch", problems=24, lo=2000, hi=60000, pick=0),
    ]


def _log(rng, lo, hi):
    return int(round(np.exp(rng.uniform(np.log(lo), np.log(hi)))))


def draw(rng):
    kind = rng.choice(["poisson", "poisson", "poisson", "assembly", "elasticity", "compliance", "batch"])
    if kind in ("poisson", "assembly"):
        if rng.random() < 0.4:
            c = dict(kind=kind, nx=_log(rng, 16, 420), ny=_log(rng, 16, 420), nz=0)
        else:
            while True:
                c = dict(kind=kind, nx=_log(rng, 9, 112), ny=_log(rng, 9, 112), nz=_log(rng, 9, 112))
                if c["nx"] * c["ny"] * c["nz"] <= 900000:
                    break
        c.update(coef=rng.random() < 0.7, distort=rng.random() < 0.4)
        c.update(mode=rng.choice(["cg", "mixed"])) if kind == "poisson" else c.update(precision=rng.choice(["fp64", "mixed"]))
        return c
    if kind == "elasticity":
        if rng.random() < 0.5:
            return dict(kind=kind, nx=_log(rng, 5, 30), ny=_log(rng, 5, 28), nz=_log(rng, 5, 26),
                        precision=rng.choice(["fp64", "mixed"]), mode="none")
        return dict(kind=kind, nx=_log(rng, 5, 12), ny=_log(rng, 5, 11), nz=_log(rng, 5, 10),
                    precision=rng.choice(["fp64", "mixed"]), mode=rng.choice(["cg", "mixed"]))
    if kind == "compliance":
        nx = _log(rng, 48, 400)
        return dict(kind=kind, nx=nx, ny=2 * max(8, int(nx * rng.uniform(0.2, 0.3))))
    return dict(kind=kind, problems=rng.randint(6, 20), lo=2000, hi=_log(rng, 8000, 50000), pick=rng.randint(1, 10**6))


# ---- meshes (topology is shared by all states of one size; coordinates are per state) -----------

def _nel(case):
    return tuple(n for n in (case["nx"], case["ny"], case.get("nz", 0)) if n)


def _displacement(nel, seed):
    """Moves of the interior nodes by up to 0.25 h per axis, in node order."""
    rng = np.random.default_rng(seed + 7919)
    shape = tuple(n + 1 for n in reversed(nel))
    d = rng.uniform(-0.25, 0.25, size=shape + (len(nel),)) / np.array(nel, dtype=np.float64)
    for ax in range(len(nel)):
        for end in (0, -1):
            sl = [slice(None)] * len(nel)
            sl[ax] = end
            d[tuple(sl)] = 0.0
    return d.reshape(-1, len(nel))


@functools.lru_cache(maxsize=2)
def _mesh(nel, right):
    ct = "Hexahedron" if len(nel) == 3 else "Quadrilateral"
    g = fa.generate_grid(ct, nel, (0.0,) * len(nel), right)
    return g, fa.create_coloring(g)


class _View:
    """A resident device array for torch.as_tensor; keeps the system that owns the memory."""

    def __init__(self, K, which):
        self.K = K
        p, n = ctypes.c_void_p(), ctypes.c_int64(0)
        K.ctx.call("fem_device_pointer", which, ctypes.byref(p), ctypes.byref(n))
        self.__cuda_array_interface__ = dict(shape=(n.value,), typestr="<f8", data=(p.value, False), version=2)


def _resident(K, which):
    t = torch.as_tensor(_View(K, which), device="cuda")
    t.owner = K      # the memory lives as long as the tensor object
    return t


def _system(nel, right, ip, qr, moved=None):
    g0, colors = _mesh(nel, right)
    g = fa.Grid(g0.celltype, g0.cells, g0.nodes if moved is None else g0.nodes + moved, g0.facetsets)
    dh = fa.DofHandler(g).add("u", ip).close(device=0)
    K = fa.allocate_matrix(fa.MI355XCSC, dh)
    f = fa.allocate_vector(K)
    cv = fa.CellValues(fa.QuadratureRule(g.refshape, qr), ip)
    return dict(g=g, dh=dh, K=K, f=f, cv=cv, colors=colors,
                nz=_resident(K, 0), fv=_resident(K, 1))


def _coef(ncells, seed):
    return np.exp(np.random.default_rng(seed).normal(0.0, 0.5, size=ncells))


def _source(seed):
    return float(np.random.default_rng(seed + 1).uniform(0.5, 2.0))


def _unit(dim):
    return (1.0,) * dim


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        b = BatchedPoisson()
        rng = np.random.default_rng(seed)
        for grid, dh, colors, ch in _batch_problems(case["problems"], case["lo"], case["hi"], case["pick"]):
            b.add(grid, dh, colors, ch, np.exp(rng.normal(0.0, 0.5, size=grid.ncells)))
        b.finalize()
        return dict(kind=kind, batch=b, u=[np.empty(p["ndofs"]) for p in b.problems])
    nel = _nel(case)
    dim = len(nel)
    if kind in ("poisson", "assembly"):
        shape = "RefHexahedron" if dim == 3 else "RefQuadrilateral"
        s = _system(nel, _unit(dim), fa.Lagrange(shape, 1), 2, _displacement(nel, seed) if case["distort"] else None)
        names = ("left", "right") if dim == 3 else ("left", "right", "bottom", "top")
        ch = fa.ConstraintHandler(s["dh"])
        ch.add(fa.Dirichlet("u", [x for n in names for x in s["g"].facetsets[n]], lambda x, t: 0.0)).close()
        s.update(kind=kind, ch=ch, el=fa.PoissonElement(k=_coef(s["g"].ncells, seed) if case["coef"] else None, source=_source(seed)),
                 mode=case.get("mode"), precision=case.get("precision", "fp64"))
        return s
    if kind == "elasticity":
        ip = fa.Lagrange("RefHexahedron", 2) ** 3
        s = _system(nel, _unit(3), ip, 3)
        ch = fa.ConstraintHandler(s["dh"])
        ch.add(fa.Dirichlet("u", s["g"].facetsets["left"], lambda x, t: [0.0, 0.0, 0.0])).close()
        E = np.random.default_rng(seed).uniform(0.5, 2.0, s["g"].ncells)
        s.update(kind=kind, ch=ch, el=fa.ElasticityElement(E=E, nu=NU), mode=case["mode"], precision=case["precision"],
                 facets=fa.FacetValues(fa.FacetQuadratureRule("RefHexahedron", 3), ip))
        return s
    ip = fa.Lagrange("RefQuadrilateral", 1) ** 2
    s = _system(nel, (2.0, 1.0), ip, 2)
    g, dh = s["g"], s["dh"]
    ch = fa.ConstraintHandler(dh)
    ch.add(fa.Dirichlet("u", g.facetsets["left"], lambda x, t: [0.0, 0.0])).close()
    # the node in the middle of the right edge: corner 3 of the cell below it
    ydof = int(dh.cell_dofs[(nel[1] // 2) * nel[0] - 1, 2 * 2 + 1])

    def loads(K, f):
        fa.add_point_load(K, f, [ydof], [-1.0])

    s.update(kind=kind, theta=_theta(nel, seed),
             problem=ComplianceProblem(s["K"], s["f"], s["cv"], s["colors"], ch, loads, EMIN, PENAL, NU, rtol=2e-9))
    return s


def _theta(nel, seed):
    return np.random.default_rng(seed).uniform(0.2, 1.0, nel[0] * nel[1])


def _batch_sizes(problems, lo, hi, pick):
    rng = np.random.default_rng(pick)
    out = []
    for i in range(problems):
        t = float(np.exp(rng.uniform(np.log(lo), np.log(hi))))
        if i % 2:
            n = max(4, int(round(t ** (1 / 3) * rng.uniform(0.8, 1.2))))
            m = max(4, int(round((t / n) ** 0.5)))
            out.append((n, m, max(4, int(t / (n * m)))))
        else:
            n = max(8, int(round(t ** 0.5 * rng.uniform(0.8, 1.2))))
            out.append((n, max(8, int(t / n))))
    return out


@functools.lru_cache(maxsize=2)
def _batch_problems(problems, lo, hi, pick):
    out = []
    for nel in _batch_sizes(problems, lo, hi, pick):
        ct = "Hexahedron" if len(nel) == 3 else "Quadrilateral"
        out.append(poisson_problem(ct, nel, np.ones(int(np.prod(nel))))[:4])
    return out


def run(s):
    kind = s["kind"]
    if kind == "batch":
        b = s["batch"]
        b.run("mixed", rtol=RTOL)
        for i, u in enumerate(s["u"]):
            b._call("fem_batch_download", i, None, None, L.ptr(u, ctypes.c_double))
        return s["u"]
    if kind == "compliance":
        J, dtheta, dX, _ = s["problem"].compliance(s["theta"])
        return dict(J=J, dtheta=dtheta, dX=dX, K=s["nz"], f=s["fv"])
    K, f = s["K"], s["f"]
    fa.assemble_global(fa.start_assemble(K, f), s["cv"], s["colors"], s["el"], precision=s["precision"])
    if kind == "elasticity":
        fa.apply_traction(K, f, s["facets"], s["g"].facetsets["right"], (0.0, 0.0, -1.0))
    fa.apply(K, f, s["ch"])
    out = dict(K=s["nz"], f=s["fv"])
    if kind == "poisson" or (kind == "elasticity" and s["mode"] != "none"):
        out["u"] = fa.solve(K, f, mode=s["mode"], rtol=RTOL, maxit=20000).u
    return out


# ---- counts --------------------------------------------------------------------------------------

def _counts(nel, order, vdim):
    """cells, nodes, dofs and pattern entries of the tensor mesh."""
    nodes = int(np.prod([n + 1 for n in nel]))
    cells = int(np.prod(nel))
    if order == 1:
        nd = nodes
        nnz = int(np.prod([3 * n + 1 for n in nel]))
    else:   # per axis: vertex couples to 5 (3 at the ends), midpoint to 3
        nd = int(np.prod([2 * n + 1 for n in nel]))
        nnz = int(np.prod([5 * (n - 1) + 6 + 3 * n for n in nel]))
    return cells, nodes, nd * vdim, nnz * vdim * vdim


def work(case):
    kind = case["kind"]
    if kind == "batch":
        by = fl = 0
        for nel in _batch_sizes(case["problems"], case["lo"], case["hi"], case["pick"]):
            cells, nodes, nd, nnz = _counts(nel, 1, 1)
            npc = 2 ** len(nel)
            by += cells * (4 * npc * 2 + 8) + 8 * nodes * len(nel) + 8 * nnz + 16 * nd
            fl += cells * npc * npc * 10 + 2 * nnz
        return dict(bytes=by, flops=fl)
    nel = _nel(case)
    order, vdim, npc = (2, 3, 27) if kind == "elasticity" else (1, 2, 4) if kind == "compliance" else (1, 1, 2 ** len(nel))
    cells, nodes, nd, nnz = _counts(nel, order, vdim)
    by = cells * (4 * 2 ** len(nel) + 4 * npc * vdim + 8) + 8 * nodes * len(nel) + 8 * nnz + 8 * nd
    fl = cells * (6 * 27 ** 3 * 2 if order == 2 else npc * npc * vdim * vdim * 10)
    if kind in ("poisson", "compliance") or case.get("mode") in ("cg", "mixed"):
        by += 8 * nd
        fl += 2 * nnz
    if kind == "compliance":
        by += 16 * cells + 16 * nodes
    return dict(bytes=by, flops=fl)


# ---- the same outputs from plain torch / numpy in 64 bits ------------------------------------------

_V3 = [(-1, -1, -1), (1, -1, -1), (1, 1, -1), (-1, 1, -1), (-1, -1, 1), (1, -1, 1), (1, 1, 1), (-1, 1, 1)]
_Q3 = _V3 + [(0, -1, -1), (1, 0, -1), (0, 1, -1), (-1, 0, -1), (0, -1, 1), (1, 0, 1), (0, 1, 1), (-1, 0, 1),
             (-1, -1, 0), (1, -1, 0), (1, 1, 0), (-1, 1, 0), (0, 0, -1), (0, -1, 0), (1, 0, 0), (0, 1, 0),
             (-1, 0, 0), (0, 0, 1), (0, 0, 0)]
_V2 = [(-1, -1), (1, -1), (1, 1), (-1, 1)]


def _basis(ref, order, pts):
    """Values [q, a] and gradients [q, a, d] of the tensor Lagrange basis at the points ref."""
    def one(c, t):
        if order == 1:
            return (1 + c * t) / 2, np.full_like(t, c / 2)
        return {-1: (t * (t - 1) / 2, t - 0.5), 1: (t * (t + 1) / 2, t + 0.5), 0: (1 - t * t, -2 * t)}[c]
    dim = pts.shape[1]
    N = np.ones((len(pts), len(ref)))
    dN = np.ones((len(pts), len(ref), dim))
    for a, r in enumerate(ref):
        vd = [one(r[d], pts[:, d]) for d in range(dim)]
        for d in range(dim):
            N[:, a] *= vd[d][0]
            for e in range(dim):
                dN[:, a, e] *= vd[d][1] if d == e else vd[d][0]
    return N, dN


def _gauss(dim, n):
    x, w = np.polynomial.legendre.leggauss(n)
    g = np.stack([a.ravel() for a in np.meshgrid(*([x] * dim), indexing="ij")], axis=1)
    return g, np.prod(np.stack([a.ravel() for a in np.meshgrid(*([w] * dim), indexing="ij")], axis=1), axis=1)


class _Exact:
    """Element arrays and the global system of one tensor mesh, dofs numbered by first visit."""

    def __init__(self, nel, right, order, vdim, moved=None):
        dim, dev = len(nel), "cuda"
        vert = np.array(_V3 if dim == 3 else _V2)
        ref = np.array(_Q3) if order == 2 else vert
        cid = np.stack([a.ravel() for a in np.meshgrid(*[np.arange(n) for n in reversed(nel)], indexing="ij")][::-1], axis=1)

        def ids(local, step):
            n = [step * m + 1 for m in nel]
            at = step * cid[:, None, :] + (local[None] + 1) * step // 2
            k = at[..., dim - 1]
            for d in range(dim - 2, -1, -1):
                k = k * n[d] + at[..., d]
            return k
        self.verts = ids(vert, 1)
        key = ids(ref, order)
        flat = key.ravel()
        _, first, inv = np.unique(flat, return_index=True, return_inverse=True)
        rank = np.empty(len(first), dtype=np.int64)
        rank[np.argsort(first, kind="stable")] = np.arange(len(first))
        self.node = rank[inv.ravel()].reshape(key.shape)          # dof node of each cell's basis function
        self.nnode, self.vdim, self.dim = len(first), vdim, dim
        self.n = self.nnode * vdim
        ax = [np.linspace(0.0, right[d], nel[d] + 1) for d in range(dim)]
        X = np.stack([a.ravel() for a in np.meshgrid(*reversed(ax), indexing="ij")][::-1], axis=1)
        X = X if moved is None else X + moved
        self.X = torch.tensor(X, device=dev)
        self.pos = torch.empty((self.nnode, dim), device=dev, dtype=torch.float64)   # positions of the dof nodes
        M, _ = _basis([tuple(v) for v in vert], 1, ref.astype(float))
        self.tv = torch.tensor(self.verts, device=dev)
        self.pos[torch.tensor(self.node, device=dev).reshape(-1)] = torch.einsum(
            "am,cmd->cad", torch.tensor(M, device=dev), self.X[self.tv]).reshape(-1, dim)
        self.dofs = torch.tensor((self.node[:, :, None] * vdim + np.arange(vdim)).reshape(len(cid), -1), device=dev)
        pts, w = _gauss(dim, 2 if order == 1 else 3)
        N, dN = _basis([tuple(r) for r in ref], order, pts)
        _, dM = _basis([tuple(v) for v in vert], 1, pts)
        self.N, self.dN, self.dM, self.w = (torch.tensor(a, device=dev) for a in (N, dN, dM, w))

    def geometry(self, cells, X=None):
        """Physical gradients [c, q, a, d] and dV [c, q] of a range of cells."""
        J = torch.einsum("cmi,qmd->cqid", (self.X if X is None else X)[self.tv[cells]], self.dM)
        G = torch.einsum("qad,cqdi->cqai", self.dN, torch.linalg.inv(J))
        return G, torch.linalg.det(J) * self.w

    def matrices(self, coef, elastic, cells, X=None):
        G, dV = self.geometry(cells, X)
        if not elastic:
            return torch.einsum("cqai,cqbi->cab", G * (dV * coef[cells, None])[:, :, None, None], G)
        lam, mu = NU / ((1 + NU) * (1 - 2 * NU)), 1 / (2 * (1 + NU))
        P = torch.einsum("cqai,cqbj->caibj", G * (dV * coef[cells, None])[:, :, None, None], G)
        tr = torch.einsum("caibi->cab", P)
        K = lam * P + mu * P.permute(0, 1, 4, 3, 2)
        for i in range(self.dim):
            K[:, :, i, :, i] += mu * tr
        return K.reshape(K.shape[0], self.dofs.shape[1], -1)

    def assemble(self, coef, elastic, source, step):
        nc, nb = self.dofs.shape
        keys, vals = torch.zeros(0, dtype=torch.int64, device="cuda"), None
        pairs = [(self.dofs[i:i + step, None, :] * self.n + self.dofs[i:i + step, :, None]).reshape(-1)
                 for i in range(0, nc, step)]
        keys = torch.unique(torch.cat([torch.unique(p) for p in pairs]))
        vals = torch.zeros(len(keys), dtype=torch.float64, device="cuda")
        f = torch.zeros(self.n, dtype=torch.float64, device="cuda")
        for i, p in zip(range(0, nc, step), pairs):
            sl = slice(i, min(nc, i + step))
            Ke = self.matrices(coef, elastic, sl)        # [c, row, col]: CSC order is (col, row), Ke symmetric
            vals.index_add_(0, torch.searchsorted(keys, p), Ke.reshape(-1))
            if source:
                fe = torch.einsum("qa,cq->ca", self.N, self.geometry(sl)[1]) * source
                f.index_add_(0, self.dofs[sl].reshape(-1), fe.reshape(-1))
        self.col, self.row = torch.div(keys, self.n, rounding_mode="floor"), keys % self.n
        return vals, f

    def constrain(self, vals, f, fixed):
        m = vals[self.row == self.col].abs().sum() / self.n
        hit = fixed[self.row] | fixed[self.col]
        vals[hit] = 0.0
        vals[(self.row == self.col) & fixed[self.row]] = m
        f[fixed] = 0.0

    def solve(self, vals, f, most):
        ptr = torch.zeros(self.n + 1, dtype=torch.int64, device="cuda")
        ptr[1:] = torch.cumsum(torch.bincount(self.col, minlength=self.n), 0)
        A = torch.sparse_csr_tensor(ptr, self.row, vals, (self.n, self.n))
        return _pcg(lambda v: A @ v, vals[self.row == self.col], f, most)


def _pcg(A, diag, f, most):
    """Jacobi CG restarted on its true residual until that no longer falls."""
    u, res = torch.zeros_like(f), f.clone()
    best = float(f.norm())
    for _ in range(4):
        x, r = torch.zeros_like(f), res.clone()
        z = r / diag
        p, rz = z.clone(), r @ z
        r0 = r.norm()
        for it in range(most):
            q = A(p)
            a = rz / (p @ q)
            x += a * p
            r -= a * q
            z = r / diag
            new = r @ z
            p = z + (new / rz) * p
            rz = new
            if it % 25 == 24 and bool(r.norm() < 1e-9 * r0):
                break
        u = u + x
        res = f - A(u)
        now = float(res.norm())
        if now > 0.3 * best or now < 2e-15 * float(f.norm()):
            break
        best = now
    return u


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        rng = np.random.default_rng(seed)
        out = []
        for nel in _batch_sizes(case["problems"], case["lo"], case["hi"], case["pick"]):
            k = np.exp(rng.normal(0.0, 0.5, size=int(np.prod(nel))))
            e = _Exact(nel, tuple(1.0 for _ in nel), 1, 1)
            e.X = e.X * 2 - 1           # generate_grid's default domain
            e.pos = e.pos * 2 - 1
            vals, f = e.assemble(torch.tensor(k, device="cuda"), False, 1.0, 1 << 19)
            e.constrain(vals, f, (e.pos.abs() > 1 - 1e-9).any(dim=1))
            out.append(e.solve(vals, f, 3000).cpu())
        return out
    nel = _nel(case)
    dim = len(nel)
    if kind in ("poisson", "assembly"):
        e = _Exact(nel, _unit(dim), 1, 1, _displacement(nel, seed) if case["distort"] else None)
        k = _coef(len(e.verts), seed) if case["coef"] else np.ones(len(e.verts))
        vals, f = e.assemble(torch.tensor(k, device="cuda"), False, _source(seed), 1 << 19)
        on = ((e.pos < 1e-9) | (e.pos > 1 - 1e-9))
        e.constrain(vals, f, on[:, 0] if dim == 3 else on.any(dim=1))
        out = dict(K=vals, f=f)
        if kind == "poisson":
            out["u"] = e.solve(vals, f, 3000).cpu()
        return out
    if kind == "elasticity":
        e = _Exact(nel, _unit(3), 2, 3)
        E = np.random.default_rng(seed).uniform(0.5, 2.0, len(e.verts))
        vals, f = e.assemble(torch.tensor(E, device="cuda"), True, 0.0, 1 << 12)
        # unit traction -z on x = 1: the face integrals of the quadratic basis are h/6 (1, 4, 1) per axis
        right = (np.arange(len(e.verts)) % nel[0]) == nel[0] - 1
        for a, r in enumerate(_Q3):
            if r[0] == 1:
                w = np.prod([(4.0 if r[d] == 0 else 1.0) / (6.0 * nel[d]) for d in (1, 2)])
                at = torch.tensor(e.node[right, a] * 3 + 2, device="cuda")
                f.index_add_(0, at, torch.full((len(at),), -w, dtype=torch.float64, device="cuda"))
        e.constrain(vals, f, (e.pos[:, 0] < 1e-9).repeat_interleave(3))
        out = dict(K=vals, f=f)
        if case["mode"] != "none":
            out["u"] = e.solve(vals, f, 8000).cpu()
        return out
    e = _Exact(nel, (2.0, 1.0), 1, 2)
    th = torch.tensor(_theta(nel, seed), device="cuda")
    E = EMIN + th ** PENAL * (1 - EMIN)
    vals, f = e.assemble(E, True, 0.0, 1 << 18)
    tip = e.node[(nel[1] // 2) * nel[0] - 1, 2]
    f[2 * tip + 1] -= 1.0
    e.constrain(vals, f, (e.pos[:, 0] < 1e-9).repeat_interleave(2))
    u = e.solve(vals, f, 9000)
    th.requires_grad_(True)
    X = e.X.clone().requires_grad_(True)
    ue = u[e.dofs]
    Ke = e.matrices(EMIN + th ** PENAL * (1 - EMIN), True, slice(None), X)
    energy = (torch.einsum("cab,cb->ca", Ke, ue) * ue).sum()
    dth, dX = torch.autograd.grad(energy, (th, X))
    return dict(J=float(f @ u), dtheta=-dth.cpu(), dX=-dX.cpu(), K=vals, f=f)
