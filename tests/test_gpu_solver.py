"""GPU GMG-PCG solver and SIMP loop against the CPU oracle (small meshes)."""
import numpy as np
import pytest

from oracle import ops as oops
from oracle import topopt as otop
from oracle.solvers import MultiGrid as OMultiGrid

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _edgeto():
    import edgeto_amd
    return edgeto_amd


def _cantilever_3d(ET, nel, nu=0.3, rmin=2.0):
    nx, ny, nz = nel
    mesh = ET.CuStructuredMesh3D(nx, ny, nz, nx, ny, nz,
                                 stiffness=lambda x0: ET.auto_stiffness(x0, 1.0, nu))
    kernel = ET.CuStructuredStiffnessKernel(mesh)
    filt = ET.CuStructuredFilter3D(mesh, rmin)
    # clamp face x = 0: node (i=0, j, k) -> j*nx1*nz1 + k
    nx1, ny1, nz1 = nx + 1, ny + 1, nz + 1
    j, k = np.meshgrid(np.arange(ny1), np.arange(nz1), indexing="ij")
    clamp = (j * nx1 * nz1 + k).ravel()
    load = np.array([0 * nx1 * nz1 + nx * nz1 + kk for kk in range(nz1)])  # x = L, y = 0 edge
    return mesh, kernel, filt, clamp, load


def _cantilever_nodes(nel):
    """Clamped face x = 0 and the loaded edge x = L, y = 0 (node ids)."""
    nx, ny, nz = nel
    nx1, ny1, nz1 = nx + 1, ny + 1, nz + 1
    j, k = np.meshgrid(np.arange(ny1), np.arange(nz1), indexing="ij")
    clamp = (j * nx1 * nz1 + k).ravel()
    load = np.array([nx * nz1 + kk for kk in range(nz1)])
    return clamp, load


def _oracle_problem(nel, nu, rmin, clamp, load, fy):
    prob = otop.Problem(nel, nu=nu, r_min=rmin)
    dof = prob.dof
    for d in range(dof):
        prob.cons[clamp * dof + d] = True
    prob.f[load * dof + 1] = fy
    return prob


# fine-grid operator variants: (ET_TUNE_WHT, ET_TUNE_MX_F32, ET_TUNE_MX_F64); None = library default
_OPS = {"default": None, "tiled": (0, 0, 0, 0, 0, 0), "matrix": (0, 1, 1, 1, 1 << 30, 1),
        "wht": (1, 0, 0, 1, 300000, 1)}
# ET_TUNE_WHT, ET_TUNE_MX_F32, ET_TUNE_MX_F64, ET_TUNE_COARSE_LIB, ET_TUNE_ROW_STENCIL_NODES,
# ET_TUNE_LEVEL1_MF
_KNOBS = (7, 3, 4, 9, 12, 13)


@pytest.fixture
def fine_ops(request):
    from edgeto_amd import _lib as L
    L.load()
    knobs = _OPS[request.param]
    old = [L.lib().et_tune_get(k) for k in _KNOBS]
    if knobs is not None:
        for k, v in zip(_KNOBS, knobs):
            L.call("et_tune_set", k, v)
    yield request.param
    for k, v in zip(_KNOBS, old):
        L.call("et_tune_set", k, v)


@pytest.mark.parametrize("fine_ops", ["default", "tiled", "matrix", "wht"], indirect=True)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nel,n_level", [((16, 8, 8), 2), ((24, 12, 12), 2)])
def test_solve_matches_direct(precision, nel, n_level, fine_ops):
    ET = _edgeto()
    mesh, kernel, filt, clamp, load = _cantilever_3d(ET, nel)
    rng = np.random.default_rng(0)
    E = rng.uniform(0.05, 1.0, mesh.n_el)
    kernel.set_rho(torch.tensor(E, device="cuda"))
    tp = ET.CuTopOpt(mesh, ET.SingleMaterial(void=1e-9, penalty=3.0, volume_fraction=0.3), kernel,
                     None, filt, verbose=False)
    tp.add_BC_nodal(clamp, np.array([[1, 1, 1]]))
    tp.add_F_nodal(load, np.array([[0.0, -1.0 / len(load), 0.0]]))
    solver = ET.CuMultiGrid(mesh, kernel, tol=1e-10, n_smooth=2, n_level=n_level, precision=precision)
    x, res = solver.solve(tp.f, use_last=False)
    assert res < 1e-10
    prob = _oracle_problem(nel, 0.3, 2.0, clamp, load, -1.0 / len(load))
    A = oops.assemble(prob.K0, prob.elements, E, prob.cons, prob.n_dof)
    import scipy.sparse.linalg as spla
    xd = spla.spsolve(A.tocsc(), prob.f)
    xg = x.cpu().numpy()
    assert np.linalg.norm(prob.f - A @ xg) / np.linalg.norm(prob.f) < 2e-10
    assert np.linalg.norm(xg - xd) / np.linalg.norm(xd) < 1e-7
    if precision == "fp64":
        # same algorithm as the oracle's GPU-semantics MultiGrid: PCG iteration counts agree
        om = OMultiGrid(prob.nel, prob.dof, tol=1e-10, n_smooth=2, n_level=n_level, mode="gpu")
        om.solve(A, prob.f, use_last=False)
        assert abs(om.last_iters - solver.last_iterations) <= 1


def test_simp_trajectory_2d():
    """Short 2-D MBB run (config-1 setup at reduced size) vs the oracle, GPU omega semantics."""
    ET = _edgeto()
    nelx, nely = 40, 20
    mesh = ET.CuStructuredMesh2D(nelx, nely, nelx, nely,
                                 stiffness=lambda x0: ET.auto_stiffness(x0, 1.0, 0.3))
    kernel = ET.CuStructuredStiffnessKernel(mesh)
    filt = ET.CuStructuredFilter2D(mesh, 1.5)
    mat = ET.SingleMaterial(void=1e-9, penalty=3.0, volume_fraction=0.5)
    solver = ET.CuMultiGrid(mesh, kernel, tol=1e-8, n_smooth=3, n_level=2)
    tp = ET.CuTopOpt(mesh, mat, kernel, solver, filt, max_iter=10, ch_tol=0, fun_tol=0, verbose=False)
    nx1 = nelx + 1
    left = np.arange(nely + 1) * nx1
    tp.add_BC_nodal(left, np.array([[1, 0]]))
    tp.add_BC_nodal(np.array([nelx]), np.array([[0, 1]]))
    tp.add_F_nodal(np.array([nely * nx1]), np.array([[0.0, -1.0]]))
    x, flag, hist = tp.optimize(save_comp_history=True, rho_init=np.full(mesh.n_el, 0.5))
    prob = otop.Problem((nelx, nely), nu=0.3, r_min=1.5)
    prob.cons[left * 2] = True
    prob.cons[nelx * 2 + 1] = True
    prob.f[nely * nx1 * 2 + 1] = -1.0
    omat = otop.SingleMaterial(void=1e-9, penalty=3.0, volume_fraction=0.5)
    osol = OMultiGrid(prob.nel, 2, tol=1e-8, n_smooth=3, n_level=2, mode="gpu")
    xo, _, ohist = otop.optimize(prob, omat, osol, np.full(prob.n_el, 0.5), 10, ch_tol=0, fun_tol=0)
    comp_gpu = np.array([tp.iteration_log[0]["comp"]] + hist["comp_history"])
    comp_ref = np.array(ohist["comp"])
    assert np.max(np.abs(comp_gpu - comp_ref) / comp_ref) < 1e-6
    assert np.max(np.abs(x.cpu().numpy() - xo)) < 1e-4


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("level1_mf", [1, 0])
@pytest.mark.parametrize("nel", [(16, 8, 8), (20, 12, 10)])
def test_level_operators_match_galerkin(precision, level1_mf, nel):
    """Every smoothing level's operator (fine grid, matrix-free or stencil first coarse level,
    stencil levels) against the oracle's Galerkin products R A R^T on a clamped cantilever with
    random densities, so the constrained-DOF correction of the first coarse level is exercised."""
    ET = _edgeto()
    from edgeto_amd import _lib as L
    old = L.lib().et_tune_get(13)
    L.call("et_tune_set", 13, level1_mf)
    try:
        mesh, kernel, filt, clamp, load = _cantilever_3d(ET, nel)
        rng = np.random.default_rng(3)
        E = rng.uniform(0.01, 1.0, mesh.n_el)
        kernel.set_rho(torch.tensor(E, device="cuda"))
        tp = ET.CuTopOpt(mesh, ET.SingleMaterial(void=1e-9, penalty=3.0, volume_fraction=0.3), kernel,
                         None, filt, verbose=False)
        tp.add_BC_nodal(clamp, np.array([[1, 1, 1]]))
        tp.add_F_nodal(load, np.array([[0.0, -1.0 / len(load), 0.0]]))
        n_level = 3
        solver = ET.CuMultiGrid(mesh, kernel, tol=1e-6, n_smooth=2, n_level=n_level, precision=precision)
        solver.solve(tp.f, use_last=False)
    finally:
        L.call("et_tune_set", 13, old)
    prob = _oracle_problem(nel, 0.3, 2.0, clamp, load, -1.0 / len(load))
    A = oops.assemble(prob.K0, prob.elements, E, prob.cons, prob.n_dof).tocsr()
    from oracle import mgm as omgm
    dt = torch.float32 if precision == "mixed" else torch.float64
    tol = 2e-5 if precision == "mixed" else 1e-11
    lnel = tuple(nel)
    for level in range(n_level):
        if level > 0:
            R = omgm.restriction_matrix(lnel, 3)
            A = (R @ A @ R.T).tocsr()
            lnel = tuple(n // 2 for n in lnel)
        x = rng.standard_normal(A.shape[0])
        xt = torch.tensor(x, dtype=dt, device="cuda")
        yt = torch.empty_like(xt)
        L.call("et_mg_apply_level", solver._handle, level, L.ptr(xt), L.ptr(yt))
        ref = A @ x
        err = np.abs(yt.cpu().numpy() - ref).max() / np.abs(ref).max()
        assert err < tol, (level, err)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nel", [(4, 4, 4), (30, 6, 8), (6, 36, 128), (8, 10, 130), (12, 8, 280), (128, 64, 64)])
def test_level1_tiles(nel, precision):
    """The matrix-free first coarse level against the stored Galerkin stencil of the same level: grids
    of one tile and of several, columns of 64 elements and more (several tiles along z), with and
    without the split by component (the largest grid), constrained DOFs on a face and inside.  Both
    sum some 200 products in different orders."""
    ET = _edgeto()
    from edgeto_amd import _lib as L
    rng = np.random.default_rng(51)
    E = rng.uniform(0.01, 1.0, int(np.prod(nel)))
    dt = torch.float32 if precision == "mixed" else torch.float64
    x = torch.tensor(rng.standard_normal(3 * int(np.prod([n // 2 + 1 for n in nel]))), dtype=dt, device="cuda")
    y = []
    old = L.lib().et_tune_get(13)
    for level1_mf in (1, 0):
        L.call("et_tune_set", 13, level1_mf)
        try:
            mesh, kernel, filt, clamp, load = _cantilever_3d(ET, nel)
            kernel.set_rho(torch.tensor(E, device="cuda"))
            tp = ET.CuTopOpt(mesh, ET.SingleMaterial(void=1e-9, penalty=3.0, volume_fraction=0.3), kernel,
                             None, filt, verbose=False)
            tp.add_BC_nodal(clamp, np.array([[1, 1, 1]]))
            tp.add_BC_nodal(np.arange(mesh.n_nodes)[7::1013], np.array([[0, 1, 0]]))
            tp.add_F_nodal(load, np.array([[0.0, -1.0 / len(load), 0.0]]))
            solver = ET.CuMultiGrid(mesh, kernel, tol=1e-30, maxiter=1, n_smooth=2, n_level=2, precision=precision)
            solver.solve(tp.f, use_last=False)
        finally:
            L.call("et_tune_set", 13, old)
        y.append(torch.empty_like(x))
        L.call("et_mg_apply_level", solver._handle, 1, L.ptr(x), L.ptr(y[-1]))
    err = ((y[0] - y[1]).abs().max() / y[1].abs().max()).item()
    assert err < (1e-5 if precision == "mixed" else 1e-13), err


@pytest.mark.parametrize("coarse_lib", [2, 1, 0])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nel", [(16, 8, 8), (24, 12, 12), (32, 16, 16)])
def test_coarse_solve_matches_dense(coarse_lib, precision, nel):
    """The coarsest-grid direct solve (band Cholesky with explicit L^-1, rocSOLVER, in-house
    dense) against a dense solve of the oracle's coarsest Galerkin operator R A R^T."""
    ET = _edgeto()
    from edgeto_amd import _lib as L
    old = L.lib().et_tune_get(9)
    L.call("et_tune_set", 9, coarse_lib)
    n_level = 2
    try:
        mesh, kernel, filt, clamp, load = _cantilever_3d(ET, nel)
        rng = np.random.default_rng(5)
        E = rng.uniform(0.01, 1.0, mesh.n_el)
        kernel.set_rho(torch.tensor(E, device="cuda"))
        tp = ET.CuTopOpt(mesh, ET.SingleMaterial(void=1e-9, penalty=3.0, volume_fraction=0.3), kernel,
                         None, filt, verbose=False)
        tp.add_BC_nodal(clamp, np.array([[1, 1, 1]]))
        tp.add_F_nodal(load, np.array([[0.0, -1.0 / len(load), 0.0]]))
        solver = ET.CuMultiGrid(mesh, kernel, tol=1e-6, n_smooth=2, n_level=n_level, precision=precision)
        solver.solve(tp.f, use_last=False)
    finally:
        L.call("et_tune_set", 9, old)
    prob = _oracle_problem(nel, 0.3, 2.0, clamp, load, -1.0 / len(load))
    A = oops.assemble(prob.K0, prob.elements, E, prob.cons, prob.n_dof).tocsr()
    from oracle import mgm as omgm
    lnel = tuple(nel)
    for _ in range(n_level):
        R = omgm.restriction_matrix(lnel, 3)
        A = (R @ A @ R.T).tocsr()
        lnel = tuple(n // 2 for n in lnel)
    b = rng.standard_normal(A.shape[0])
    xd = np.linalg.solve(A.toarray(), b)
    dt = torch.float32 if precision == "mixed" else torch.float64
    bt = torch.tensor(b, dtype=dt, device="cuda")
    xt = torch.empty_like(bt)
    L.call("et_mg_coarse_solve", solver._handle, L.ptr(bt), L.ptr(xt))
    err = np.abs(xt.cpu().numpy() - xd).max() / np.abs(xd).max()
    assert err < (1e-5 if precision == "mixed" else 1e-9), err


def _pcg_run(precision, maxiter, fused_rz, strict=False):
    """One solve of a clamped 24x12x12 cantilever with random densities under ET_TUNE_FUSED_RZ."""
    ET = _edgeto()
    from edgeto_amd import _lib as L
    nel = (24, 12, 12)
    old = L.lib().et_tune_get(14)
    L.call("et_tune_set", 14, fused_rz)
    try:
        mesh, kernel, filt, clamp, load = _cantilever_3d(ET, nel)
        rng = np.random.default_rng(11)
        E = rng.uniform(0.05, 1.0, mesh.n_el)
        kernel.set_rho(torch.tensor(E, device="cuda"))
        tp = ET.CuTopOpt(mesh, ET.SingleMaterial(void=1e-9, penalty=3.0, volume_fraction=0.3), kernel,
                         None, filt, verbose=False)
        tp.add_BC_nodal(clamp, np.array([[1, 1, 1]]))
        tp.add_F_nodal(load, np.array([[0.0, -1.0 / len(load), 0.0]]))
        solver = ET.CuMultiGrid(mesh, kernel, tol=1e-10, maxiter=maxiter, n_smooth=2, n_level=2,
                                precision=precision, strict=strict)
        x, res = solver.solve(tp.f, use_last=False)
        iters = solver.last_iterations
    finally:
        L.call("et_tune_set", 14, old)
    prob = _oracle_problem(nel, 0.3, 2.0, clamp, load, -1.0 / len(load))
    A = oops.assemble(prob.K0, prob.elements, E, prob.cons, prob.n_dof)
    xg = x.cpu().numpy()
    true_res = np.linalg.norm(prob.f - A @ xg) / np.linalg.norm(prob.f)
    return iters, res, true_res, xg


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("maxiter", [1000, 7])
def test_pcg_vector_updates(precision, maxiter):
    """PCG with r.z summed inside the last fine-grid sweep (ET_TUNE_FUSED_RZ = 1) and by its own
    pass (0), and with x += alpha p deferred to the p update: the returned x must satisfy
    |f - A x| / |f| = the reported residual, whether the loop ends on the tolerance or on
    maxiter, and both settings give the same iterates."""
    runs = []
    for fused_rz in (1, 0):
        iters, res, true_res, xg = _pcg_run(precision, maxiter, fused_rz)
        if maxiter == 7:
            assert iters == 7
            assert res > 1e-10
        else:
            assert iters < maxiter and res < 1e-10
        # the recursively updated residual tracks the true one
        assert abs(true_res - res) <= 1e-6 * res + 2e-11, (fused_rz, true_res, res)
        runs.append((iters, xg))
    (i0, x0), (i1, x1) = runs
    assert abs(i0 - i1) <= 1
    if i0 == i1:
        tol = 1e-6 if precision == "mixed" else 1e-9
        assert np.linalg.norm(x0 - x1) / np.linalg.norm(x0) < tol


def test_pcg_maxiter_status():
    """maxiter reached above the tolerance: et_mg_solve returns ET_ENOCONV; MultiGrid(strict=True)
    raises it, strict=False returns the last iterate and its residual."""
    from edgeto_amd import _lib as L
    with pytest.raises(L.EdgetoError) as ei:
        _pcg_run("fp64", 7, 1, strict=True)
    assert ei.value.status == L.ET_ENOCONV
    iters, res, true_res, _ = _pcg_run("fp64", 7, 1, strict=False)
    assert iters == 7 and res > 1e-10


@pytest.mark.parametrize("nel", [(96, 48, 12), (72, 48, 16), (48, 36, 28), (36, 32, 40), (28, 28, 60)])
def test_tile_operator_with_the_transformed_basis(nel):
    """The one-shot tile operator as the FP64 solver uses it from 50 000 nodes, one to four element
    columns per wavefront: the fine-grid product against the oracle (rows of 192 products), and three
    PCG iterations against the marching operator's for one to three sweeps, with r.z summed in the
    last sweep and apart from it (every mode of the V-cycle; other summation orders)."""
    ET = _edgeto()
    from edgeto_amd import _lib as L
    rng = np.random.default_rng(61)
    E = rng.uniform(0.05, 1.0, int(np.prod(nel)))
    mesh, kernel, filt, clamp, load = _cantilever_3d(ET, nel)
    kernel.set_rho(torch.tensor(E, device="cuda"))
    tp = ET.CuTopOpt(mesh, ET.SingleMaterial(void=1e-9, penalty=3.0, volume_fraction=0.3), kernel, None, filt,
                     verbose=False)
    tp.add_BC_nodal(clamp, np.array([[1, 1, 1]]))
    tp.add_F_nodal(load, np.array([[0.0, -1.0 / len(load), 0.0]]))
    assert mesh.n_nodes >= 50000  # below, the solver keeps the marching operator
    xs, old = {}, (L.lib().et_tune_get(18), L.lib().et_tune_get(14))
    try:
        for n_smooth in (1, 2, 3):
            for rz in (1, 0):
                for nodes in (old[0], 0):
                    L.call("et_tune_set", 18, nodes)
                    L.call("et_tune_set", 14, rz)
                    solver = ET.CuMultiGrid(mesh, kernel, tol=1e-30, maxiter=3, n_smooth=n_smooth, n_level=2)
                    xs[nodes] = solver.solve(tp.f, use_last=False)[0]
                    if nodes and n_smooth == 2 and rz:
                        x = torch.tensor(rng.standard_normal(kernel.shape[0]), device="cuda")
                        y = torch.empty_like(x)
                        L.call("et_mg_apply_level", solver._handle, 0, L.ptr(x), L.ptr(y))
                        prob = _oracle_problem(nel, 0.3, 2.0, clamp, load, -1.0 / len(load))
                        ref = oops.matvec(prob.K0, prob.elements, E, x.cpu().numpy(), prob.cons)
                        assert np.abs(y.cpu().numpy() - ref).max() < 1e-13 * np.abs(ref).max()
                err = ((xs[old[0]] - xs[0]).norm() / xs[0].norm()).item()
                assert 0 < err < 1e-12, (n_smooth, rz, err)  # 0: the same operator twice
    finally:
        L.call("et_tune_set", 18, old[0])
        L.call("et_tune_set", 14, old[1])


# (ET_TUNE_WHT_THREADS_F32, ET_TUNE_WHT_THREADS_F64, ET_TUNE_WHT_SLICES_F32, ET_TUNE_WHT_SLICES_F64)
_TILES = {"default": (1024, 512, 16, 8), "f32_half": (512, 512, 8, 8), "f64_full": (1024, 512, 16, 16),
          "f64_256": (1024, 256, 16, 8)}


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_solve_tile_variants(precision):
    """The V-cycle's fused fine-grid modes (two zero-guess sweeps in one pass, the last sweep with
    the r.z partials) on every transformed-basis tile shape: the solution of a clamped cantilever
    with random densities against a direct solve, and each iteration count against the default
    tile's."""
    ET = _edgeto()
    from edgeto_amd import _lib as L
    import scipy.sparse.linalg as spla
    knobs = (10, 11, 15, 16)
    nel = (24, 12, 12)
    prob = _oracle_problem(nel, 0.3, 2.0, *_cantilever_nodes(nel), -1.0 / (nel[2] + 1))
    rng = np.random.default_rng(17)
    E = rng.uniform(0.05, 1.0, int(np.prod(nel)))
    A = oops.assemble(prob.K0, prob.elements, E, prob.cons, prob.n_dof)
    xd = spla.spsolve(A.tocsc(), prob.f)
    iters = {}
    for tiles, values in _TILES.items():
        old = [L.lib().et_tune_get(k) for k in knobs]
        for k, v in zip(knobs, values):
            L.call("et_tune_set", k, v)
        try:
            mesh, kernel, filt, clamp, load = _cantilever_3d(ET, nel)
            kernel.set_rho(torch.tensor(E, device="cuda"))
            tp = ET.CuTopOpt(mesh, ET.SingleMaterial(void=1e-9, penalty=3.0, volume_fraction=0.3), kernel,
                             None, filt, verbose=False)
            tp.add_BC_nodal(clamp, np.array([[1, 1, 1]]))
            tp.add_F_nodal(load, np.array([[0.0, -1.0 / len(load), 0.0]]))
            solver = ET.CuMultiGrid(mesh, kernel, tol=1e-10, n_smooth=2, n_level=2, precision=precision)
            x, res = solver.solve(tp.f, use_last=False)
            iters[tiles] = solver.last_iterations
        finally:
            for k, v in zip(knobs, old):
                L.call("et_tune_set", k, v)
        assert res < 1e-10, tiles
        xg = x.cpu().numpy()
        assert np.linalg.norm(xg - xd) / np.linalg.norm(xd) < 1e-7, tiles
    for tiles, it in iters.items():
        assert abs(iters["default"] - it) <= 1, (tiles, iters)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nel,n_level", [((2, 2), 1), ((15, 9), 1), ((16, 16), 2), ((17, 33), 2), ((33, 18), 3),
                                         ((62, 46), 2), ((96, 16), 3)])
def test_fused_2d_cycle(nel, n_level, precision):
    """2-D V(2,2) cycles (each leg of a level in one kernel) at the edges of their 16 x 16 node tiles,
    with odd extents on any level and single constrained DOFs inside the grid: the iterate after five
    PCG iterations (six cycles) against the oracle's.  Odd extents do not converge further with this
    hierarchy, so the iterate is compared, not a solution.  A cycle's rounding is some 100 units in
    the last place, and an early CG iterate amplifies it by at most the 10 to 100 fold of its residual's
    ups and downs: 1e-11 and, with an FP32 cycle, 2e-3."""
    ET = _edgeto()
    mesh = ET.CuStructuredMesh2D(*nel, *nel, stiffness=lambda x0: ET.auto_stiffness(x0, 1.0, 0.3))
    kernel = ET.CuStructuredStiffnessKernel(mesh)
    rng = np.random.default_rng(41)
    E = rng.uniform(0.3, 1.0, mesh.n_el)
    kernel.set_rho(torch.tensor(E, device="cuda"))
    tp = ET.CuTopOpt(mesh, ET.SingleMaterial(void=1e-9, penalty=3.0, volume_fraction=0.3), kernel,
                     None, ET.CuStructuredFilter2D(mesh, 1.5), verbose=False)
    nx1, n_nodes = nel[0] + 1, (nel[0] + 1) * (nel[1] + 1)
    clamp = np.arange(nel[1] + 1) * nx1
    roller = np.arange(n_nodes)[4::37]  # one component fixed, tile interiors and borders
    load = n_nodes - 1
    tp.add_BC_nodal(clamp, np.array([[1, 1]]))
    tp.add_BC_nodal(roller, np.array([[0, 1]]))
    tp.add_F_nodal(np.array([load]), np.array([[1.0, 0.0]]))
    solver = ET.CuMultiGrid(mesh, kernel, tol=1e-30, maxiter=5, n_smooth=2, n_level=n_level, precision=precision,
                            strict=False)
    x, res = solver.solve(tp.f, use_last=False)
    prob = otop.Problem(nel, nu=0.3, r_min=1.5)
    prob.cons[clamp * 2] = prob.cons[clamp * 2 + 1] = prob.cons[roller * 2 + 1] = True
    prob.f[2 * load] = 1.0
    A = oops.assemble(prob.K0, prob.elements, E, prob.cons, prob.n_dof)
    om = OMultiGrid(nel, 2, tol=1e-30, maxiter=5, n_smooth=2, n_level=n_level, mode="gpu")
    xo, ores = om.solve(A, prob.f, use_last=False)
    assert om.last_iters == solver.last_iterations == 5
    err = np.linalg.norm(x.cpu().numpy() - xo) / np.linalg.norm(xo)
    print(nel, n_level, precision, err, abs(res - ores) / ores)
    assert err < (1e-11 if precision == "fp64" else 2e-3)


@pytest.mark.parametrize("w_level", [0, 1, [0, 1]])
def test_fused_2d_cycle_beside_w_levels(w_level):
    """2-D W-cycles: levels visited twice take one kernel per operation, the others the fused legs.
    The iterate after five PCG iterations against the oracle's (bound as in test_fused_2d_cycle)."""
    ET = _edgeto()
    nel = (48, 32)
    mesh = ET.CuStructuredMesh2D(*nel, *nel, stiffness=lambda x0: ET.auto_stiffness(x0, 1.0, 0.3))
    kernel = ET.CuStructuredStiffnessKernel(mesh)
    rng = np.random.default_rng(43)
    E = rng.uniform(0.3, 1.0, mesh.n_el)
    kernel.set_rho(torch.tensor(E, device="cuda"))
    tp = ET.CuTopOpt(mesh, ET.SingleMaterial(void=1e-9, penalty=3.0, volume_fraction=0.3), kernel,
                     None, ET.CuStructuredFilter2D(mesh, 1.5), verbose=False)
    clamp, load = np.arange(nel[1] + 1) * (nel[0] + 1), (nel[0] + 1) * (nel[1] + 1) - 1
    tp.add_BC_nodal(clamp, np.array([[1, 1]]))
    tp.add_F_nodal(np.array([load]), np.array([[1.0, 0.0]]))
    args = dict(tol=1e-30, maxiter=5, n_smooth=2, n_level=3, cycle="w", w_level=w_level)
    solver = ET.CuMultiGrid(mesh, kernel, strict=False, **args)
    x, _ = solver.solve(tp.f, use_last=False)
    prob = otop.Problem(nel, nu=0.3, r_min=1.5)
    prob.cons[clamp * 2] = prob.cons[clamp * 2 + 1] = True
    prob.f[2 * load] = 1.0
    A = oops.assemble(prob.K0, prob.elements, E, prob.cons, prob.n_dof)
    om = OMultiGrid(nel, 2, mode="gpu", **{**args, "w_level": np.atleast_1d(w_level).tolist()})
    xo, _ = om.solve(A, prob.f, use_last=False)
    assert om.last_iters == solver.last_iterations == 5
    assert np.linalg.norm(x.cpu().numpy() - xo) / np.linalg.norm(xo) < 1e-11


def test_mixed_2d_iterations():
    """An ill-conditioned 2-D solve (moduli over two decades, more than 100 PCG iterations): the FP32
    V-cycle costs no iterations while r.z is summed with r in FP64 (with r's FP32 copy: a quarter
    more).  A tenth is left for the cycle's own rounding."""
    ET = _edgeto()
    nel = (352, 96)
    mesh = ET.CuStructuredMesh2D(*nel, *nel, stiffness=lambda x0: ET.auto_stiffness(x0, 1.0, 0.3))
    kernel = ET.CuStructuredStiffnessKernel(mesh)
    rng = np.random.default_rng(7)
    X, Y = np.meshgrid(np.linspace(0, 1, nel[0]), np.linspace(0, 1, nel[1]), indexing="ij")
    f = sum(np.sin(2 * np.pi * (rng.uniform(-3, 3) * X + rng.uniform(-6, 6) * Y + rng.uniform())) for _ in range(8))
    kernel.set_rho(torch.tensor((0.5 + 0.35 * np.tanh(f)).ravel() ** 3, device="cuda"))
    tp = ET.CuTopOpt(mesh, ET.SingleMaterial(void=1e-9, penalty=3.0, volume_fraction=0.3), kernel,
                     None, ET.CuStructuredFilter2D(mesh, 1.5), verbose=False)
    tp.add_BC_nodal(np.arange(nel[1] + 1) * (nel[0] + 1), np.array([[1, 0]]))
    tp.add_BC_nodal(np.array([nel[0]]), np.array([[0, 1]]))
    tp.add_F_nodal(np.array([nel[1] * (nel[0] + 1)]), np.array([[0.0, -1.0]]))
    iters = {}
    for precision in ("fp64", "mixed"):
        solver = ET.CuMultiGrid(mesh, kernel, tol=1e-8, n_smooth=2, n_level=4, precision=precision)
        _, res = solver.solve(tp.f, use_last=False)
        assert res < 1e-8
        iters[precision] = solver.last_iterations
    print(iters)
    assert iters["mixed"] <= 1.1 * iters["fp64"], iters


@pytest.mark.parametrize("nel", [(16, 8), (8, 4, 4), (12, 6, 6)])
@pytest.mark.parametrize("method", ["cg", "gmres"])
def test_krylov_solvers(nel, method):
    """CuCG / CuGMRES (unpreconditioned, matrix-free) against the oracle's restatement of the
    cupyx iterations on the same clamped problem: iteration counts, the reported true residual
    and the solution."""
    ET = _edgeto()
    from oracle import krylov
    from oracle import mesh as omesh
    dim = len(nel)
    if dim == 3:
        mesh, kernel, filt, clamp, load = _cantilever_3d(ET, nel)
        fvec = np.array([[0.0, -1.0 / len(load), 0.0]])
    else:
        mesh = ET.CuStructuredMesh2D(*nel, *nel, stiffness=lambda x0: ET.auto_stiffness(x0, 1.0, 0.3))
        kernel = ET.CuStructuredStiffnessKernel(mesh)
        filt = ET.CuStructuredFilter2D(mesh, 1.5)
        clamp = np.arange(nel[1] + 1) * (nel[0] + 1)
        load = np.array([nel[0]])
        fvec = np.array([[0.0, -1.0]])
    rng = np.random.default_rng(21)
    E = rng.uniform(0.2, 1.0, mesh.n_el)
    kernel.set_rho(torch.tensor(E, device="cuda"))
    tp = ET.CuTopOpt(mesh, ET.SingleMaterial(void=1e-9, penalty=3.0, volume_fraction=0.3), kernel,
                     None, filt, verbose=False)
    tp.add_BC_nodal(clamp, np.ones((1, dim), dtype=np.int64))
    tp.add_F_nodal(load, fvec)
    tol = 1e-8
    solver = (ET.CuCG if method == "cg" else ET.CuGMRES)(kernel, maxiter=20000, tol=tol)
    x, res = solver.solve(tp.f, use_last=False)
    cons = kernel.constraints.cpu().numpy()
    f = tp.f.cpu().numpy()
    el = omesh.elements_3d(*nel) if dim == 3 else omesh.elements_2d(*nel)
    A = oops.assemble(mesh.K_single_host, el, E, cons, kernel.shape[0])
    xg = x.cpu().numpy()
    true_res = np.linalg.norm(f - A @ xg) / np.linalg.norm(f)
    assert res <= tol and abs(true_res - res) <= 1e-3 * res
    if method == "cg":
        xo, it = krylov.cg(lambda v: A @ v, f, tol=tol, maxiter=20000)
        # rounding moves the stopping iteration of a long CG run by a few at most
        assert abs(solver.last_iterations - it) <= max(2, it // 100), (solver.last_iterations, it)
    else:
        xo, it = krylov.gmres(lambda v: A @ v, f, tol=tol, restart=20, maxiter=20000)
        assert abs(solver.last_iterations - it) <= 20, (solver.last_iterations, it)
    import scipy.sparse.linalg as spla
    xd = spla.spsolve(A.tocsc(), f)
    assert np.linalg.norm(xg - xd) / np.linalg.norm(xd) < 1e-5
    # warm start from the previous solution: converged at once
    x2, res2 = solver.solve(tp.f, use_last=True)
    assert res2 <= tol
