"""Timed cases of the SIMP path on one GPU: the calls a user's optimisation loop makes.

Kinds (each case is one public call, or the two directions of one operator):

    filter   density filter and its transpose (CuStructuredFilter2D / 3D)
    dot      structured stiffness operator times a vector, FP64
    grad     fused SIMP sensitivity with the filter transpose (the backward of the loop)
    oc       optimality-criteria design update
    solve    GMG-PCG solve of one density field, from a zero start
    simp     one whole OC iteration: design update, filter, SIMP map, solve, compliance, sensitivity
    cg       CuCG on a tetrahedral mesh: assembly of the operator and the iterations
    batch    many independent problems through the batched engine

Densities are smooth random grey designs as they occur early in a run (material between 15 %
and 85 %, so moduli span two decades: the solves take about as many iterations as those of the
cantilever benchmark); grids of the solves halve evenly down to their coarsest level; loads and supports are a clamped cantilever in
3-D and a half MBB beam in 2-D.  exact() restates every kind in plain torch, FP64.
"""
import functools
import math
import os
import sys
import time

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "edge-to_amd"))
import edgeto_amd as ET  # noqa: E402

VOID, PENAL, NU, VF, MOVE = 1e-9, 3.0, 0.3, 0.3, 0.2


def listed():
    return [
        # the filter of a small 2-D design: two launches, nothing but latency
        dict(name="filter_2d_small", kind="filter", nx=120, ny=40, nz=0, rmin=1.5),
        # the filter of a large 3-D design, the radius of the cantilever benchmark
        dict(name="filter_3d_large", kind="filter", nx=256, ny=128, nz=128, rmin=2.0),
        # one operator product on an odd, ragged 3-D grid (any Krylov loop of a user's own)
        dict(name="dot_3d_odd", kind="dot", nx=97, ny=45, nz=51),
        # one operator product on a large 2-D grid
        dict(name="dot_2d_large", kind="dot", nx=1024, ny=512, nz=0),
        # sensitivity of a mid-size 3-D design
        dict(name="grad_3d", kind="grad", nx=128, ny=64, nz=64, rmin=2.0),
        # design update of a small 2-D design
        dict(name="oc_2d_small", kind="oc", nx=120, ny=40, nz=0),
        # a small 2-D solve: the 120 x 40 half MBB beam, FP64
        dict(name="solve_2d_small", kind="solve", nx=120, ny=40, nz=0, precision="fp64", tol=1e-8),
        # a large 2-D solve, mixed precision
        dict(name="solve_2d_large", kind="solve", nx=512, ny=256, nz=0, precision="mixed", tol=1e-8),
        # an FP64 3-D solve on extents that are no powers of two (coarsest grid 15 x 7 x 6)
        dict(name="solve_3d_ragged", kind="solve", nx=120, ny=56, nz=48, precision="fp64", tol=1e-8),
        # one SIMP iteration at 12.8 M unknowns, mixed precision
        dict(name="simp_3d_large", kind="simp", nx=256, ny=128, nz=128, precision="mixed", rmin=2.0, tol=1e-8),
        # conjugate gradients on an unstructured tetrahedral mesh
        dict(name="cg_tets", kind="cg", nx=32, ny=16, nz=16, tol=1e-5),
        # a batch of small independent problems, one OC iteration each
        dict(name="batch_small", kind="batch", problems=8, longest=64, iterations=1),
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["filter", "dot", "grad", "oc", "solve", "solve", "simp", "simp", "cg", "batch"])
    if kind == "cg":
        n = _size(rng, 4, 16)
        return dict(kind=kind, nx=2 * n + rng.randint(0, 1), ny=n, nz=rng.randint(max(2, n // 2), n), tol=1e-5)
    if kind == "batch":
        return dict(kind=kind, problems=rng.randint(2, 8), longest=rng.randint(16, 64), iterations=rng.randint(1, 2))
    c = dict(kind=kind)
    small = kind in ("solve", "simp")
    if rng.random() < 0.5:
        c.update(nx=_size(rng, 32, 512 if small else 1024), ny=_size(rng, 16, 256 if small else 512), nz=0)
    else:
        n = _size(rng, 8, 64 if small else 128)
        c.update(nx=rng.randint(n, 2 * n), ny=rng.randint(max(8, n // 2), n), nz=rng.randint(max(8, n // 2), n))
    if small:
        # grids that a multigrid user picks: every level but the coarsest has even extents
        m = (4 if c["nx"] < 40 else 8) if c["nz"] else (4 if c["nx"] < 128 else 8 if c["nx"] < 256 else 16)
        c.update({a: max(8, c[a] // m * m) for a in ("nx", "ny", "nz") if c[a]})
        c.update(precision=rng.choice(["fp64", "mixed"]), tol=rng.choice([1e-6, 1e-8]))
    if kind in ("filter", "grad", "simp"):
        c["rmin"] = round(rng.uniform(1.2, 3.5), 2)
    return c


# ------------------------------------------------------------------- inputs ---

def _nel(case):
    return tuple(case[a] for a in ("nx", "ny", "nz") if case[a])


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _smooth(shape, g, waves=10):
    """Sum of random low-frequency plane waves on a grid, zero mean and unit deviation."""
    out = torch.zeros(shape, dtype=torch.float64, device="cuda")
    for _ in range(waves):
        k = (torch.rand(len(shape), generator=g, device="cuda", dtype=torch.float64) * 2 - 1) * 6 * math.pi
        phase = torch.rand(1, generator=g, device="cuda", dtype=torch.float64) * 2 * math.pi
        arg = phase
        for a, n in enumerate(shape):
            x = torch.linspace(0, n / max(shape), n, dtype=torch.float64, device="cuda")
            arg = arg + (k[a] * x).reshape([-1 if b == a else 1 for b in range(len(shape))])
        out += torch.cos(arg)
    out -= out.mean()
    return out / out.std().clamp_min(1e-12)


def _design(shape, g):
    """A grey design: values in [0.15, 0.85], mean about the volume fraction's order."""
    return (0.15 + 0.7 * torch.sigmoid(1.5 * _smooth(shape, g) - 1.0)).reshape(-1)


def _sensitivity(shape, rho, g):
    """-dc/dx as strain energies spread: positive, over several decades."""
    return -3.0 * rho ** 2 * torch.exp(1.5 * _smooth(shape, g).reshape(-1))


def _vector(nel, g):
    """A displacement-like nodal field: smooth in every component, with 1 % noise; node order
    y, x(, z), components interleaved."""
    shape = (nel[1] + 1, nel[0] + 1) + tuple(n + 1 for n in nel[2:])
    u = torch.stack([_smooth(shape, g) for _ in nel], dim=-1).reshape(-1)
    return u + 0.01 * torch.randn(u.shape, generator=g, device="cuda", dtype=torch.float64)


def _supports(nel):
    """(nodes, flags) pairs of the supports and the loaded nodes."""
    if len(nel) == 2:
        nx, ny = nel
        left = np.arange(ny + 1) * (nx + 1)
        return [(left, [1, 0]), (np.array([nx]), [0, 1])], np.array([ny * (nx + 1)])
    nx, ny, nz = nel
    j, k = np.meshgrid(np.arange(ny + 1), np.arange(nz + 1), indexing="ij")
    clamp = (j * (nx + 1) * (nz + 1) + k).ravel()
    return [(clamp, [1, 1, 1])], nx * (nz + 1) + np.arange(nz + 1)


def _load(nel, seed):
    """Total load of one unit downwards with a seeded sideways part, per loaded node."""
    r = np.random.RandomState(int(seed) % (1 << 31))
    _, nodes = _supports(nel)
    v = np.concatenate([[0.1 * r.uniform(-1, 1), -1.0], 0.1 * r.uniform(-1, 1, len(nel) - 2)])
    return nodes, v[None, :] / len(nodes)


def _mesh(nel):
    cls = ET.CuStructuredMesh2D if len(nel) == 2 else ET.CuStructuredMesh3D
    return cls(*nel, *nel, stiffness=lambda x0: ET.auto_stiffness(x0, 1.0, NU))


def _filter(mesh, rmin):
    return (ET.CuStructuredFilter2D if len(mesh.nel) == 2 else ET.CuStructuredFilter3D)(mesh, rmin)


def _kernel(mesh, nel):
    kernel = ET.CuStructuredStiffnessKernel(mesh)
    for nodes, flags in _supports(nel)[0]:
        for d, on in enumerate(flags):
            if on:
                kernel.add_constraints(nodes * len(nel) + d)
    return kernel


def _material():
    return ET.SingleMaterial(void=VOID, penalty=PENAL, volume_fraction=VF)


def _tets(nel):
    """Kuhn tetrahedra (six per cell) of a grid of unit cells: nodes, element lists."""
    nx, ny, nz = nel
    nodes = np.stack(np.meshgrid(*(np.arange(n + 1.0) for n in nel), indexing="ij"), -1).reshape(-1, 3)
    nid = np.arange(nodes.shape[0]).reshape(nx + 1, ny + 1, nz + 1)
    c = [nid[:-1, :-1, :-1], nid[1:, :-1, :-1], nid[1:, 1:, :-1], nid[:-1, 1:, :-1],
         nid[:-1, :-1, 1:], nid[1:, :-1, 1:], nid[1:, 1:, 1:], nid[:-1, 1:, 1:]]
    kuhn = [(0, 1, 2, 6), (0, 2, 3, 6), (0, 3, 7, 6), (0, 7, 4, 6), (0, 4, 5, 6), (0, 5, 1, 6)]
    return nodes, np.stack([np.stack([c[a].reshape(-1) for a in t], 1) for t in kuhn], 1).reshape(-1, 4)


@functools.lru_cache(maxsize=1)
def _tet_mesh(nel):
    """The mesh file a user's program has loaded (seconds of host work; the same for every seed)."""
    nodes, els = _tets(nel)
    return ET.CuGeneralMesh(nodes, els, stiffness=ET.AutoStiffness(1.0, NU)), nodes


def _batch_problems(case, seed):
    """Cantilevers of mixed dimension and size, half of them 2-D, one to four point loads each."""
    r = np.random.RandomState(int(seed) % (1 << 31))
    # the sizes belong to the case, not to the seed
    sizes = np.random.RandomState(case["problems"] * 1000 + case["longest"])
    out = []
    for i in range(case["problems"]):
        n = max(16, int(case["longest"] * sizes.uniform(0.5, 1.0))) // 8 * 8
        if i % 2 == 0:
            nel = (4 * n, 2 * n)
            clamp = np.arange(nel[1] + 1) * (nel[0] + 1)
            side = clamp + nel[0]
        else:
            nel = (n, n // 2, n // 2)
            plane = (nel[0] + 1) * (nel[2] + 1)
            clamp = (np.arange(nel[1] + 1)[:, None] * plane + np.arange(nel[2] + 1)[None, :]).ravel()
            side = clamp + nel[0] * (nel[2] + 1)
        loads = r.choice(side, size=int(r.randint(1, 5)), replace=False)
        dirs = r.standard_normal((len(loads), len(nel)))
        dirs /= np.linalg.norm(dirs, axis=1, keepdims=True)
        out.append(dict(dim=len(nel), nel=nel, clamp=clamp, loads=loads, dirs=dirs, vf=float(r.uniform(0.3, 0.5)),
                        rmin=float(r.uniform(1.2, 3.0)), penal=PENAL))
    return out


def _inputs(case, seed):
    """The seeded arrays of a case, shared by prepare() and exact()."""
    kind, nel, g = case["kind"], _nel(case), _gen(seed)
    if kind == "filter":
        rho = _design(nel, g)
        return dict(x=rho, v=_sensitivity(nel, rho, g))
    if kind == "dot":
        return dict(E=_design(nel, g) ** PENAL, u=_vector(nel, g))
    if kind == "grad":
        return dict(xt=_design(nel, g), U=_vector(nel, g))
    if kind == "oc":
        rho = _design(nel, g)
        return dict(rho=rho, df=_sensitivity(nel, rho, g))
    if kind == "solve":
        return dict(E=_design(nel, g) ** PENAL)
    if kind == "simp":
        rho = _design(nel, g)
        return dict(rho=rho, df=_sensitivity(nel, rho, g))
    shape = nel + (6,)
    return dict(E=_design(shape, g) ** PENAL)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return dict(kind=kind, batch=ET.BatchTopOpt(_batch_problems(case, seed), precision="mixed"),
                    iterations=case["iterations"], n=case["problems"])
    nel = _nel(case)
    s = dict(kind=kind, **_inputs(case, seed))
    if kind == "cg":
        mesh, nodes = _tet_mesh(nel)
        kernel = ET.CuGeneralStiffnessKernel(mesh)
        solver = ET.CuCG(kernel, maxiter=5000, tol=case["tol"])
        tp = ET.CuTopOpt(mesh, _material(), kernel, solver, None, verbose=False)
        tp.add_BC_nodal(np.nonzero(nodes[:, 0] == 0.0)[0], np.array([[1, 1, 1]]))
        end = np.nonzero((nodes[:, 0] == nel[0]) & (nodes[:, 1] == 0.0))[0]
        tp.add_F_nodal(end, _load(nel, seed)[1] * (nel[2] + 1) / len(end))
        kernel._pattern()  # the sparsity pattern is built once per mesh
        return dict(s, solver=solver, f=tp.f)
    mesh = _mesh(nel)
    if kind == "filter":
        return dict(s, filt=_filter(mesh, case["rmin"]))
    kernel = _kernel(mesh, nel)
    if kind == "dot":
        kernel.set_rho(s["E"])
        return dict(s, kernel=kernel)
    if kind == "grad":
        return dict(s, kernel=kernel, filt=_filter(mesh, case["rmin"]))
    if kind == "oc":
        return dict(s, tp=ET.CuTopOpt(mesh, _material(), kernel, ET.CuCG(kernel), None, move=MOVE, verbose=False))
    solver = ET.CuMultiGrid(mesh, kernel, tol=case["tol"], n_smooth=2, n_level=ET.gmg_levels(nel),
                            precision=case["precision"])
    filt = _filter(mesh, case["rmin"]) if kind == "simp" else None
    # reuse_sol=False: every pass solves from a zero start, so that a pass repeats
    tp = ET.CuTopOpt(mesh, _material(), kernel, solver, filt, move=MOVE, reuse_sol=False, verbose=False)
    tp.add_F_nodal(*_load(nel, seed))
    return dict(s, tp=tp, solver=solver, f=tp.f)


def run(s):
    kind = s["kind"]
    if kind == "filter":
        return s["filt"].dot(s["x"]), s["filt"].T.dot(s["v"])
    if kind == "dot":
        return s["kernel"].dot(s["u"])
    if kind == "grad":
        return s["filt"].simp_adjoint(s["kernel"], s["U"], s["xt"], PENAL, VOID)
    if kind == "oc":
        return s["tp"].update_design(s["rho"], s["df"])
    if kind in ("solve", "cg"):
        return s["solver"].solve(s["f"], rho=s["E"], use_last=False)[0]
    if kind == "simp":
        rho = s["tp"].update_design(s["rho"], s["df"])
        comp, df, _ = s["tp"].solve_and_process(rho, 1)
        return dict(rho=rho, compliance=comp, df=df)
    out = s["batch"].run(s["iterations"])
    return dict(compliance=[p["compliance"] for p in out["problems"]],
                design=[s["batch"].design(i) for i in range(s["n"])])


# ------------------------------------------------------ necessary work, bounds ---

# PCG iterations that the algorithm (V(2,2) cycles) takes on these designs, for work() only
ITER_2D, ITER_3D, ITER_CG = 60, 120, 1500


def _solve_work(nel, precision, iters):
    """One GMG-PCG solve: per iteration the FP64 product and vector updates, and a V(2,2) cycle
    whose fine sweeps each read their operands and write their result once."""
    dim = len(nel)
    ne, nd = math.prod(nel), dim * math.prod(n + 1 for n in nel)
    t = 4 if precision == "mixed" else 8
    levels = 8 / 7 if dim == 3 else 4 / 3
    per = 8 * (10 * nd + ne) + t * (18 * nd + 4 * ne) * levels
    flops = ne * (260 if dim == 3 else 64) * (1 + 5 * levels) + 40 * nd
    return iters * per, iters * flops


def work(case):
    kind = case["kind"]
    if kind == "batch":
        b = f = 0
        for p in _batch_problems(case, 0):
            w = _solve_work(p["nel"], "mixed", ITER_2D if p["dim"] == 2 else ITER_3D)
            b, f = b + w[0] * (1 + case["iterations"]), f + w[1] * (1 + case["iterations"])
        return dict(bytes=b, flops=f)
    nel = _nel(case)
    dim, ne = len(nel), math.prod(nel)
    nd = dim * math.prod(n + 1 for n in nel)
    taps = math.pi * case.get("rmin", 1) ** 2 if dim == 2 else 4.19 * case.get("rmin", 1) ** 3
    if kind == "filter":
        return dict(bytes=8 * 4 * ne, flops=4 * taps * ne)
    if kind == "dot":
        return dict(bytes=8 * (2 * nd + ne) + nd, flops=ne * (260 if dim == 3 else 64))
    if kind == "grad":
        return dict(bytes=8 * (nd + 2 * ne), flops=ne * (160 + 2 * taps))
    if kind == "oc":
        return dict(bytes=8 * 3 * ne, flops=10 * ne)
    if kind == "cg":
        ne, nnz = 6 * ne, 41 * nd  # the assembled rows of a Kuhn mesh average 41 entries
        return dict(bytes=8 * 144 * ne + ITER_CG * (12 * nnz + 8 * 10 * nd), flops=ITER_CG * (2 * nnz + 10 * nd))
    b, f = _solve_work(nel, case["precision"], ITER_2D if dim == 2 else ITER_3D)
    if kind == "simp":
        b, f = b + 8 * (nd + 10 * ne), f + ne * (160 + 4 * taps)
    return dict(bytes=b, flops=f)


def tolerance(case):
    kind = case["kind"]
    # about four times the largest distance to exact() seen over listed and drawn cases
    if kind in ("filter", "dot", "oc"):
        return {"rel": 2e-14, "max": 1e-12}  # FP64 sums in another order
    if kind == "grad":
        return {"rel": 3e-13}  # smooth fields: the energies cancel two digits
    if kind == "cg":
        return {"rel": 2e-6}  # stops at a residual of 1e-5
    if kind == "batch":
        return {"rel": 1e-6}
    return {"rel": 10 * case["tol"]}


# ----------------------------------------------------------- plain references ---

def _q4():
    """Unit-square Q4, plane stress, E = 1 (2 x 2 Gauss)."""
    D = np.array([[1, NU, 0], [NU, 1, 0], [0, 0, (1 - NU) / 2]]) / (1 - NU * NU)
    X = np.array([[0, 0], [1, 0], [1, 1], [0, 1.0]])
    K = np.zeros((8, 8))
    for a in (-1, 1):
        for b in (-1, 1):
            p = (1 + np.array([a, b]) / math.sqrt(3)) / 2
            dN = np.array([[(2 * c[0] - 1) * (p[1] if c[1] else 1 - p[1]),
                            (2 * c[1] - 1) * (p[0] if c[0] else 1 - p[0])] for c in X])
            B = np.zeros((3, 8))
            B[0, 0::2], B[1, 1::2], B[2, 0::2], B[2, 1::2] = dN[:, 0], dN[:, 1], dN[:, 1], dN[:, 0]
            K += B.T @ D @ B / 4
    return K


_CUBE = np.array([[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0], [0, 0, 1], [1, 0, 1], [1, 1, 1], [0, 1, 1.0]])


def _strain3(dN):
    """6 x 3n strain matrix of nodal gradients dN (..., n, 3)."""
    n = dN.shape[-2]
    B = np.zeros(dN.shape[:-2] + (6, 3 * n))
    for d in range(3):
        B[..., d, d::3] = dN[..., d]
    for row, (p, q) in zip((3, 4, 5), ((0, 1), (1, 2), (0, 2))):
        B[..., row, p::3], B[..., row, q::3] = dN[..., q], dN[..., p]
    return B


def _elastic3():
    C = np.zeros((6, 6))
    C[:3, :3] = NU
    C[range(3), range(3)] = 1 - NU
    C[range(3, 6), range(3, 6)] = (1 - 2 * NU) / 2
    return C / ((1 + NU) * (1 - 2 * NU))


def _h8():
    """Unit-cube H8, E = 1 (2 x 2 x 2 Gauss)."""
    D, K = _elastic3(), np.zeros((24, 24))
    for a in (-1, 1):
        for b in (-1, 1):
            for c in (-1, 1):
                p = (1 + np.array([a, b, c]) / math.sqrt(3)) / 2
                N = np.where(_CUBE > 0, p, 1 - p)
                s = 2 * _CUBE - 1
                dN = np.stack([s[:, d] * N[:, (d + 1) % 3] * N[:, (d + 2) % 3] for d in range(3)], 1)
                B = _strain3(dN)
                K += B.T @ D @ B / 8
    return K


def _grid_elements(nel):
    """Corner nodes of every element (element order x, y(, z); node order y, x(, z))."""
    i = torch.arange(nel[0], device="cuda").reshape(-1, 1, 1)
    j = torch.arange(nel[1], device="cuda").reshape(1, -1, 1)
    if len(nel) == 2:
        k, nz, corners = torch.zeros(1, 1, 1, dtype=torch.long, device="cuda"), 1, [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0)]
    else:
        k, nz = torch.arange(nel[2], device="cuda").reshape(1, 1, -1), nel[2] + 1
        corners = [tuple(int(v) for v in c) for c in _CUBE]
    return torch.stack([(((j + b) * (nel[0] + 1) + i + a) * nz + k + c).reshape(-1) for a, b, c in corners], 1)


class _Elements:
    """sum_e E_e K_e in plain torch: K one matrix for all elements, or one per element."""

    def __init__(self, elements, K, E, fixed):
        dof = K.shape[-1] // elements.shape[1]
        self.dofs = (elements[:, :, None] * dof + torch.arange(dof, device="cuda")).reshape(elements.shape[0], -1)
        self.K, self.E, self.fixed = K, E, fixed

    def product(self, u):
        return (u[self.dofs] @ self.K) if self.K.dim() == 2 else torch.bmm(self.K, u[self.dofs][:, :, None])[:, :, 0]

    def apply(self, u):
        um = torch.where(self.fixed, 0.0, u)
        y = torch.zeros_like(u).index_add_(0, self.dofs.reshape(-1), (self.product(um) * self.E[:, None]).reshape(-1))
        return torch.where(self.fixed, u, y)

    def energy(self, u):
        return (self.product(u) * u[self.dofs]).sum(1)

    def diagonal(self):
        d = torch.diagonal(self.K, dim1=-2, dim2=-1)
        y = torch.zeros(self.fixed.numel(), dtype=torch.float64, device="cuda")
        y.index_add_(0, self.dofs.reshape(-1), (d * self.E[:, None]).reshape(-1))
        return torch.where(self.fixed, 1.0, y)

    def solve(self, b, tol=1e-13, seconds=15.0):
        """Jacobi-preconditioned CG to a residual far below any case's; None when it takes too long."""
        dinv, x, r = 1.0 / self.diagonal(), torch.zeros_like(b), b.clone()
        z = dinv * r
        p, rz, t0, nb = z.clone(), torch.dot(r, z), time.monotonic(), float(b.norm())
        for it in range(1, 200000):
            q = self.apply(p)
            alpha = rz / torch.dot(p, q)
            x += alpha * p
            r -= alpha * q
            z = dinv * r
            rz, old = torch.dot(r, z), rz
            p = z + (rz / old) * p
            if it % 50 == 0:
                if float(r.norm()) < tol * nb:
                    return x
                if time.monotonic() - t0 > seconds:
                    return None
        return None


def _fixed(nel):
    m = torch.zeros(len(nel) * math.prod(n + 1 for n in nel), dtype=torch.bool, device="cuda")
    for nodes, flags in _supports(nel)[0]:
        for d, on in enumerate(flags):
            if on:
                m[torch.as_tensor(nodes * len(nel) + d, device="cuda")] = True
    return m


def _force(nel, seed):
    f = torch.zeros(len(nel) * math.prod(n + 1 for n in nel), dtype=torch.float64, device="cuda")
    nodes, v = _load(nel, seed)
    for d in range(len(nel)):
        f[torch.as_tensor(nodes * len(nel) + d, device="cuda")] = float(v[0, d])
    return f


def _hat(nel, rmin):
    n = int(math.ceil(rmin))
    ax = torch.arange(-n, n + 1, dtype=torch.float64, device="cuda")
    d2 = sum((ax ** 2).reshape([-1 if b == a else 1 for b in range(len(nel))]) for a in range(len(nel)))
    return torch.clamp(rmin - torch.sqrt(d2), min=0.0)


def _convolve(x, w):
    """Zero-padded correlation with the (symmetric) weights, tap by tap."""
    n = (w.shape[0] - 1) // 2
    p = torch.nn.functional.pad(x, (n, n) * x.dim())
    out = torch.zeros_like(x)
    for t in (w > 0).nonzero().tolist():
        out += w[tuple(t)] * p[tuple(slice(a, a + s) for a, s in zip(t, x.shape))]
    return out


def _filtered(x, nel, rmin):
    w = _hat(nel, rmin)
    return (_convolve(x.reshape(nel), w) / _convolve(torch.ones(nel, dtype=torch.float64, device="cuda"), w)).reshape(-1)


def _filtered_t(v, nel, rmin):
    w = _hat(nel, rmin)
    return _convolve(v.reshape(nel) / _convolve(torch.ones(nel, dtype=torch.float64, device="cuda"), w), w).reshape(-1)


def _updated(rho, df):
    """The OC step by plain bisection."""
    xu, xl = (rho + MOVE).clamp(0, 1), (rho - MOVE).clamp(0, 1)
    p = (rho * torch.sqrt(torch.clamp(-df, min=0.0))).clamp_min(1e-12)
    l1, l2 = 1e-9, 1e9
    while (l2 - l1) / (l2 + l1) > 1e-4:
        mid = 0.5 * (l1 + l2)
        x = torch.maximum(xl, torch.minimum(xu, p / mid)).clamp(0, 1)
        if float(x.mean()) <= VF:
            l2 = mid
        else:
            l1 = mid
    return x


def _adjoint(op, U, xt, nel, rmin):
    return _filtered_t(-PENAL * xt.clamp(VOID, 1.0) ** (PENAL - 1) * op.energy(U), nel, rmin)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return None
    nel, s = _nel(case), _inputs(case, seed)
    if kind == "filter":
        return _filtered(s["x"], nel, case["rmin"]), _filtered_t(s["v"], nel, case["rmin"])
    if kind == "oc":
        return _updated(s["rho"], s["df"])
    if kind == "cg":
        nodes, els = _tets(nel)
        x = nodes[els]
        grad = np.linalg.inv(np.concatenate([np.ones(x.shape[:2] + (1,)), x], 2))[:, 1:, :].transpose(0, 2, 1)
        vol = np.abs(np.linalg.det(x[:, 1:] - x[:, :1])) / 6
        B = _strain3(grad)
        K = np.einsum("eia,ij,ejb->eab", B, _elastic3(), B, optimize=True) * vol[:, None, None]
        fixed = torch.as_tensor(np.repeat(nodes[:, 0] == 0.0, 3), device="cuda")
        f = torch.zeros(3 * len(nodes), dtype=torch.float64, device="cuda")
        end = np.nonzero((nodes[:, 0] == nel[0]) & (nodes[:, 1] == 0.0))[0]
        for d in range(3):
            f[torch.as_tensor(3 * end + d, device="cuda")] = float(_load(nel, seed)[1][0, d] * (nel[2] + 1) / len(end))
        return _Elements(torch.as_tensor(els, device="cuda"), torch.as_tensor(K, device="cuda"), s["E"], fixed).solve(f)
    if kind in ("solve", "simp") and math.prod(nel) > 500000:
        return None
    K = torch.as_tensor(_q4() if len(nel) == 2 else _h8(), device="cuda")
    op = _Elements(_grid_elements(nel), K, s.get("E"), _fixed(nel))
    if kind == "dot":
        return op.apply(s["u"])
    if kind == "grad":
        return _adjoint(op, s["U"], s["xt"], nel, case["rmin"])
    if kind == "solve":
        return op.solve(_force(nel, seed))
    rho = _updated(s["rho"], s["df"])
    xt = _filtered(rho, nel, case["rmin"])
    op.E = (xt ** PENAL).clamp(VOID, 1.0)
    f = _force(nel, seed)
    U = op.solve(f)
    if U is None:
        return None
    return dict(rho=rho, compliance=float(torch.dot(f, U)), df=_adjoint(op, U, xt, nel, case["rmin"]).reshape(-1, 1))
