"""The aggregation multigrid preconditioner (setup "preconditioner" =
"multigrid") on the GPU: every Krylov method and precision reaches the FP64
true relative residual 1e-8 and agrees with a direct solve (scipy splu) within
cond(A) * 1.5e-8; the hierarchy coarsens down to the dense limit; the
preconditioner cuts the iteration count against ILU(0) alone; K and V cycles,
damped-Jacobi and ILU(0) smoothing of the coarse levels, nested levels and the
dense last level (register and global-memory inverses) are all exercised;
repeated solves are bit-identical."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from phase_amd import meshgen as G
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _case(oracle, sigma, cells=6000, seed=7):
    xy, cptr, cind = H.delaunay_case(cells, 32, seed=seed)
    m, (rp, ci, v), b, g, bc = H.pressure_system(oracle, xy, cptr, cind, sigma=sigma)
    A = H.compact_sorted(rp, ci, v)
    S = (-A).tocsc()
    lmax = spla.eigsh(S, k=1, which="LA", return_eigenvectors=False)[0]
    lmin = spla.eigsh(S, k=1, sigma=0.0, which="LM", return_eigenvectors=False)[0]
    return rp, ci, v, b, A, lmax / lmin, spla.splu(A.tocsc()).solve(b)


@pytest.fixture(scope="module")
def sys1(oracle):
    return _case(oracle, 1.0)


@pytest.fixture(scope="module")
def sys2(oracle):
    return _case(oracle, 2.0, seed=8)


def _solve(hip, rp, ci, v, b, **kw):
    s = hip.HipSparseMatrixSolver(0, tolerance=1e-8, maxIters=20000, **kw)
    s.set(rp, ci, v)
    s.set_rhs(b)
    rel = s.solve()
    return s, rel, s.x()


def _check(A, b, x, x_ref, kappa, rel):
    assert rel <= 1e-8
    assert np.linalg.norm(b - A @ x) <= 1.5e-8 * np.linalg.norm(b)
    assert np.linalg.norm(x - x_ref) <= kappa * 1.5e-8 * np.linalg.norm(x_ref)


@pytest.mark.parametrize("dense", [256, 16])   # 16: nested ILU levels before the dense one
@pytest.mark.parametrize("mode,solver", [("fp64", "cg"), ("mixed", "cg"), ("fp64", "bicgstab"),
                                         ("mixed", "bicgstab")])
@pytest.mark.parametrize("which", ["sys1", "sys2"])
def test_multigrid_matches_direct(hip, request, which, mode, solver, dense):
    rp, ci, v, b, A, kappa, x_ref = request.getfixturevalue(which)
    s, rel, x = _solve(hip, rp, ci, v, b, mode=mode, solver=solver, preconditioner="multigrid",
                       multigridDenseRows=dense, multigridCoarseRows=4 if dense < 64 else 16)
    _check(A, b, x, x_ref, kappa, rel)
    lv = s.multigrid_levels()
    assert lv[0] == len(b) and lv[-1] <= dense and len(lv) >= 2
    assert all(a > c for a, c in zip(lv, lv[1:]))
    if dense < 64:
        assert len(lv) >= 4
    ilu, _, _ = _solve(hip, rp, ci, v, b, mode=mode, solver=solver)
    assert 3 * s.n_iters() <= ilu.n_iters(), (s.n_iters(), ilu.n_iters())


@pytest.mark.parametrize("smoother", ["jacobi", "ilu"])
@pytest.mark.parametrize("cycle", ["K", "V"])
def test_multigrid_cycles_converge(hip, sys2, cycle, smoother):
    rp, ci, v, b, A, kappa, x_ref = sys2
    kw = dict(multigridJacobiFrom=64) if smoother == "ilu" else {}
    s, rel, x = _solve(hip, rp, ci, v, b, mode="fp64", solver="cg", preconditioner="multigrid",
                       multigridCycle=cycle, multigridDenseRows=16, multigridCoarseRows=4, **kw)
    _check(A, b, x, x_ref, kappa, rel)


# (fine aggregate rows, coarse aggregate rows, dense limit) -> last level of
# 26, 74, 176 and 254 rows on this mesh (CPU hierarchy of the same orderings)
@pytest.mark.parametrize("pivoting", ["auto", "always"])
@pytest.mark.parametrize("fine,coarse,dense,lo,hi", [(32, 16, 60, 1, 64), (32, 4, 120, 65, 128),
                                                     (48, 16, 256, 129, 192), (32, 16, 256, 193, 256)])
def test_multigrid_dense_inverse(hip, sys1, fine, coarse, dense, lo, hi, pivoting):
    """The last level's inverse, from each register layout of the Gauss-Jordan
    kernels (up to 64, 128 and 192 rows; without pivoting, as a pressure
    system takes, and with pivoting) and from the global-memory one (above
    192): times the last level's Galerkin matrix it gives the identity to
    rounding, and the solve converges."""
    rp, ci, v, b, A, kappa, x_ref = sys1
    s, rel, x = _solve(hip, rp, ci, v, b, mode="fp64", solver="cg", preconditioner="multigrid",
                       blockRows=fine, multigridDenseRows=dense, multigridCoarseRows=coarse,
                       multigridDensePivoting=pivoting)
    _check(A, b, x, x_ref, kappa, rel)
    m, inv = s.multigrid_coarsest()
    n = len(m)
    assert lo <= n <= hi and np.abs(m).max() > 0, n
    k = np.linalg.cond(m)
    assert np.abs(inv @ m - np.eye(n)).max() <= 1e-13 * k, (n, k)
    print("dense level", n, "cond %.3g" % k, flush=True)


@pytest.mark.parametrize("n,half,rows,coarse", [(200, 1, 64, 64), (333, 7, 64, 64), (5000, 5, 64, 8), (4099, 2, 7, 7),
                                                (257, 3, 2, 64)])
def test_galerkin_sums_exact(hip, n, half, rows, coarse):
    """Coarse operators of a graph Laplacian plus 3 I with whole-number weights:
    every sum is exact, so on the dense level, through all levels above it, the
    matrix is symmetric, its entries are whole, each row sums to 3 times the
    rows it stands for, and those add up to n.  Lists of one entry and of some
    hundreds, none a multiple of the entries read together."""
    rng = np.random.default_rng(n)
    off = [sp.diags(-rng.integers(1, 9, n - d).astype(float), d) for d in range(1, half + 1)]
    up = sum(off[1:], off[0])
    A = up + up.T
    A = (A + sp.diags(3. - np.asarray(A.sum(axis=1)).ravel())).tocsr()
    A.sort_indices()
    s = hip.HipSparseMatrixSolver(0, preconditioner="multigrid", solver="cg", mode="fp64", blockRows=rows,
                                  multigridCoarseRows=coarse, multigridDenseRows=64)
    s.set(A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data)
    b = rng.standard_normal(n)
    s.set_rhs(b)
    s.solve()
    m, _ = s.multigrid_coarsest()
    sums = m.sum(axis=1) / 3.
    assert np.array_equal(m, m.T) and np.array_equal(m, np.rint(m))
    assert np.array_equal(sums, np.rint(sums)) and sums.min() >= 1. and sums.sum() == n


def test_multigrid_device_assembly_brick_aggregates(hip, oracle):
    """A device-assembled pressure equation: the solver knows the centroids,
    so every level's aggregates are bricks; the solution agrees with the
    oracle's assembly and a direct solve."""
    xy, cptr, cind = H.delaunay_case(20000, 64, seed=9)
    om = oracle.Mesh(xy, cptr, cind)
    hm = hip.HipMesh(xy, cptr, cind)
    f = om.faces()
    pid = G.boundary_patch(f["lnode"], f["rnode"], f["rcell"], xy)
    bc = np.where(pid == 2, hip.BC_FIXED, hip.BC_NORMAL_GRADIENT).astype(np.int32)
    g = G.lognormal_face_coeffs(om.n_faces, 1.0, seed=2)
    b = G.zero_mean_normal(om.n_cells, seed=3)
    e = oracle.laplacian(om, 3, gamma_face=g, bc_type=bc, phi_face=np.zeros(om.n_faces))
    e.eq(b)
    rp, ci, v, rhs = e.get()
    A = H.compact_sorted(rp, ci, v)
    x_ref = spla.spsolve(A.tocsc(), -rhs)
    for mode in ("fp64", "mixed"):
        s = hip.HipSparseMatrixSolver(0, tolerance=1e-8, maxIters=5000, mode=mode, solver="cg",
                                      preconditioner="multigrid", multigridDenseRows=64)
        s.assemble_laplacian(hm, 3, gamma_face=g, bc_type=bc, phi_face=np.zeros(om.n_faces))
        s.sub_rhs(b)
        assert s.solve() <= 1e-8
        x = s.x()
        assert np.linalg.norm(-rhs - A @ x) <= 1.5e-8 * np.linalg.norm(rhs)
        assert np.linalg.norm(x - x_ref) <= 1e-3 * np.linalg.norm(x_ref)
        assert len(s.multigrid_levels()) >= 3


def test_multigrid_repeated_solves_bit_identical(hip, sys1):
    rp, ci, v, b, A, kappa, x_ref = sys1
    out = []
    for _ in range(2):
        s, rel, x = _solve(hip, rp, ci, v, b, mode="mixed", solver="cg", preconditioner="multigrid",
                           multigridDenseRows=16, multigridCoarseRows=4)
        out.append((x, s.n_iters()))
        s.set_rhs(b)
        s.set_guess(np.zeros(len(b)))
        s.solve()
        out.append((s.x(), s.n_iters()))
    for x, it in out[1:]:
        assert np.array_equal(x, out[0][0]) and it == out[0][1]


def test_multigrid_values_change_between_solves(hip, sys1):
    """New values on the same pattern rebuild the coarse matrices and factors."""
    rp, ci, v, b, A, kappa, x_ref = sys1
    s = hip.HipSparseMatrixSolver(0, tolerance=1e-8, maxIters=5000, mode="fp64", solver="cg",
                                  preconditioner="multigrid", multigridDenseRows=16, multigridCoarseRows=4)
    for scale in (1.0, 3.0):
        s.set(rp, ci, v * scale)
        s.set_rhs(b)
        s.set_guess(np.zeros(len(b)))
        assert s.solve() <= 1e-8
        assert np.linalg.norm(b - scale * (A @ s.x())) <= 1.5e-8 * np.linalg.norm(b)


def test_multigrid_graph_aggregates_wide_coarse_rows(hip, oracle):
    """Host CSR input (no centroids: graph aggregates at every level).  At this
    size a coarse level has rows that couple to more rows of their own or of
    later ILU blocks than the sweep kernels keep in registers, so the sweeps'
    remaining-entry loops run; the solve still reaches the FP64 goal in a
    multigrid iteration count."""
    xy, cptr, cind = H.delaunay_case(250000, 128, seed=14)
    m, (rp, ci, v), b, g, bc = H.pressure_system(oracle, xy, cptr, cind, sigma=1.0)
    A = H.compact_sorted(rp, ci, v)
    for mode in ("fp64", "mixed"):
        s, rel, x = _solve(hip, rp, ci, v, b, mode=mode, solver="cg", preconditioner="multigrid",
                           multigridJacobiFrom=64)  # ILU(0) sweeps on every coarse level
        assert rel <= 1e-8
        assert np.linalg.norm(b - A @ x) <= 1.5e-8 * np.linalg.norm(b)
        assert len(s.multigrid_levels()) >= 4
        assert s.n_iters() <= 150, s.n_iters()


@pytest.mark.parametrize("cycle", ["K", "V"])
@pytest.mark.parametrize("nx,rows,coarse", [(128, 1, 16), (170, 1, 16), (180, 2, 16), (250, 3, 16), (300, 3, 16),
                                            (303, 4, 16), (350, 4, 16), (360, 5, 16), (170, 1, 4), (230, 2, 8),
                                            (250, 3, 6)])
def test_last_levels_match_direct(hip, oracle, nx, rows, coarse, cycle):
    """The level above the dense one in one workgroup, at 1 to 3 rows per thread
    (565 to about 3,000 rows, 979 and 1,100 at the edges; graph aggregates,
    whose rows are partly wider than the entries held in registers), and as
    launches above that (3,087 to 4,316 rows) and over more than 256 dense rows
    (2,110 over 370; 979 over 254 and 1,785 over 237 below the line).  A solve to 1e-10 is within
    cond(A) 1e-10 of the direct one; cond(A) is below 16 nx^2 for these
    coefficients (8 / pi^2 nx^2 times the spread e^(4 sigma) within four
    deviations, sigma = 0.5).  A wrong coarse correction shows in the iteration
    count: K cycles take 38 to 42, V cycles twice that."""
    m, (rp, ci, v), b, g, bc = H.pressure_system(oracle, *G.rectilinear(nx, nx), sigma=0.5)
    A = H.compact_sorted(rp, ci, v)
    x_ref = spla.splu(A.tocsc()).solve(b)
    for mode in ("fp64", "mixed"):
        s = hip.HipSparseMatrixSolver(0, tolerance=1e-10, maxIters=2000, solver="cg", mode=mode,
                                      preconditioner="multigrid", multigridDenseRows=512, multigridCycle=cycle,
                                      multigridCoarseRows=coarse)
        s.set(rp, ci, v)
        s.set_rhs(b)
        s.solve()
        x = s.x()
        lv = s.multigrid_levels()
        assert (lv[-2] + 1023) // 1024 == rows, lv
        assert np.linalg.norm(x - x_ref) <= 16 * nx * nx * 1e-10 * np.linalg.norm(x_ref)
        assert s.n_iters() <= (60 if cycle == "K" else 130)
        s.zero_guess()
        s.solve()
        assert np.array_equal(s.x(), x)


@pytest.mark.parametrize("nx,ny", [(512, 512), (513, 512)])
@pytest.mark.parametrize("mode", ["fp64", "mixed"])
def test_prolongation_forms_match_known(hip, oracle, nx, ny, mode):
    """Up to 2^18 rows the finest level's prolongation runs with the post-smoothing
    residual, above apart from it.  A solve for a known field reaches its goal in
    the usual number of iterations and is within cond(A) 1e-10 of the field,
    cond(A) below 16 nx^2 as in the tests below."""
    m, (rp, ci, v), b, g, bc = H.pressure_system(oracle, *G.rectilinear(nx, ny), sigma=0.5)
    x_ref = np.random.default_rng(nx).standard_normal(nx * ny)
    s = hip.HipSparseMatrixSolver(0, tolerance=1e-10, maxIters=2000, solver="cg", mode=mode,
                                  preconditioner="multigrid")
    s.set(rp, ci, v)
    s.set_rhs(oracle.spmv(rp, ci, v, x_ref))
    s.solve()
    x = s.x()
    assert np.linalg.norm(x - x_ref) <= 16 * nx * nx * 1e-10 * np.linalg.norm(x_ref)
    assert s.n_iters() <= 60, s.n_iters()
    s.zero_guess()
    s.solve()
    assert np.array_equal(s.x(), x)


@pytest.mark.parametrize("mode,most", [("fp64", 208), ("mixed", 242)])
def test_multigrid_memory(hip, mode, most):
    """Device memory a first multigrid solve of 2^19 rows takes: Krylov and cycle
    vectors, factors and hierarchy, 204 bytes a row in FP64 and 236 mixed (in
    whole 2 MB; the rows' five entries are set before).  A vector that nothing
    reads would be 8 bytes more, 12 in mixed mode."""
    def free():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.load_library().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    def solver(n):
        off = [sp.diags(-np.ones(n - d), d) for d in (1, 2)]
        up = off[0] + off[1]
        A = up + up.T
        A = (A + sp.diags(3. - np.asarray(A.sum(axis=1)).ravel())).tocsr()
        s = hip.HipSparseMatrixSolver(0, solver="cg", mode=mode, preconditioner="multigrid", maxIters=3)
        s.set(A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data)
        s.set_rhs(np.ones(n))
        return s

    solver(5000).solve(raise_on_noconv=False)  # the kernels are loaded
    n = 1 << 19
    s = solver(n)
    before = free()
    s.solve(raise_on_noconv=False)
    taken = before - free()
    assert taken <= most * n, taken / n


@pytest.mark.parametrize("solver", ["bicgstab", "gmres"])
@pytest.mark.parametrize("nx,rows,coarse,lo,hi", [(128, 1, 16, 1, 256), (170, 1, 16, 1, 256), (180, 2, 16, 1, 256),
                                                  (250, 3, 16, 1, 256), (230, 2, 4, 257, 512)])
def test_last_levels_ilu_match_direct(hip, oracle, nx, rows, coarse, lo, hi, solver):
    """As above with ILU(0)-smoothed coarse levels: V cycles under BiCGStab, K
    cycles under GMRES; 565 to 1,100 rows in one workgroup (block inverses),
    2,110 as launches, and 1,785 over more than 256 dense rows."""
    m, (rp, ci, v), b, g, bc = H.pressure_system(oracle, *G.rectilinear(nx, nx), sigma=0.5)
    A = H.compact_sorted(rp, ci, v)
    x_ref = spla.splu(A.tocsc()).solve(b)
    for mode in ("fp64", "mixed"):
        s = hip.HipSparseMatrixSolver(0, tolerance=1e-10, maxIters=2000, solver=solver, mode=mode,
                                      preconditioner="multigrid", multigridCoarseRows=coarse, multigridDenseRows=hi)
        s.set(rp, ci, v)
        s.set_rhs(b)
        s.solve()
        x = s.x()
        lv = s.multigrid_levels()
        assert (lv[1] + 1023) // 1024 == rows and lo <= lv[2] <= hi, lv
        assert np.linalg.norm(x - x_ref) <= 16 * nx * nx * 1e-10 * np.linalg.norm(x_ref)
        assert s.n_iters() <= 200
        s.zero_guess()
        s.solve()
        assert np.array_equal(s.x(), x)
