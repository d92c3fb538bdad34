"""GPU parity of the sparse solver through the C ABI (libphase_hip.so).

Bit-exact: SpMV (same per-row order, fused multiply-add chain) and the ILU(0)
factor (same IKJ update order) against the FP64 oracle on the same inputs.
Tolerance: solved fields, relative residual <= 1e-8 (FP64 true residual) and
agreement with a direct (scipy splu) solution within cond-scaled bounds.
"""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from tests import helpers as H

pytestmark = pytest.mark.gpu


def _solver(hip, **kw):
    s = hip.HipSparseMatrixSolver(0)
    for k, v in kw.items():
        s.setup(k, v)
    return s


@pytest.fixture(scope="module")
def tri_case(oracle):
    xy, cptr, cind = H.delaunay_case(6000, 32, seed=7)
    m, (rp, ci, v), b, g, bc = H.pressure_system(oracle, xy, cptr, cind, sigma=1.0)
    return rp, ci, v, b


def test_spmv_bitwise(hip, oracle, tri_case):
    rp, ci, v, b = tri_case
    s = _solver(hip)
    s.set(rp, ci, v)
    x = np.random.default_rng(1).standard_normal(len(rp) - 1)
    y = s.spmv(x)
    assert np.array_equal(y, oracle.spmv(rp, ci, v, x))
    y32 = s.spmv(x, single=True)
    ref = oracle.spmv(rp, ci, v, x)
    assert np.max(np.abs(y32 - ref)) <= 1e-5 * np.max(np.abs(ref))


def test_ilu_factor_bitwise(hip, oracle, tri_case):
    rp, ci, v, b = tri_case
    s = _solver(hip)
    s.set(rp, ci, v)
    perm, frp, fci, fv = s.ilu_export()
    A = H.permuted(H.compact_sorted(rp, ci, v), perm)
    fac = oracle.ilu0(A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data)
    assert np.array_equal(frp, A.indptr)
    assert np.array_equal(fci, A.indices)
    assert np.array_equal(fv, fac)


@pytest.mark.parametrize("n,half,block_rows", [(1, 0, 64), (64, 1, 64), (65, 7, 64), (333, 7, 64), (333, 7, 7),
                                               (1000, 3, 64), (257, 5, 1), (129, 2, 33)])
def test_ilu_factor_row_widths_bitwise(hip, oracle, n, half, block_rows):
    """Rows of up to 2 * half + 1 entries with a fifth of them missing (an
    unsymmetric pattern, empty couplings in between): more and fewer entries,
    and more and fewer updates of an entry, than the factor kernel reads ahead;
    whole and part blocks.  Same update order as the oracle: equal bits."""
    rng = np.random.default_rng(n + half)
    rp, ci, v = [0], [], []
    for i in range(n):
        c = [j for j in range(max(0, i - half), min(n, i + half + 1)) if j == i or rng.random() < 0.8]
        a = rng.standard_normal(len(c))
        a[c.index(i)] = 2.0 * half + 4.0
        ci += c
        v += list(a)
        rp.append(len(ci))
    rp, ci, v = np.array(rp, np.int32), np.array(ci, np.int32), np.array(v)
    s = _solver(hip, blockRows=block_rows)
    s.set(rp, ci, v)
    perm, frp, fci, fv = s.ilu_export()
    A = H.permuted(H.compact_sorted(rp, ci, v), perm)
    fac = oracle.ilu0(A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data)
    assert np.array_equal(frp, A.indptr)
    assert np.array_equal(fci, A.indices)
    assert np.array_equal(fv, fac)


@pytest.mark.parametrize("per_colour,half", [(4096, 3), (4097, 3), (4097, 5), (5120, 3), (5121, 3), (5121, 5),
                                             (8192, 3), (8193, 3)])
def test_sweep_forms_by_blocks(hip, per_colour, half):
    """The sweeps' backward levels change their form with the blocks of a launch
    (FP64: fused above 4,096, the other colour between 5,121 and 8,192).  One
    GMRES step from zero leaves x = alpha M^-1 b: every row of L U x must be alpha
    b to the round-off of two substitutions, gamma_k |L||U||x| with k the rows'
    entries (at most 6 and 6) and a few roundings of the step's scalings."""
    rows = 33  # more than half a block: one aggregate per block
    n = 2 * per_colour * rows
    rng = np.random.default_rng(per_colour)
    offs = range(-half, half + 1)
    A = sp.diags([rng.uniform(-1.0, 1.0, n - abs(d)) + (12.0 if d == 0 else 0.0) for d in offs], offs).tocsr()
    b = rng.standard_normal(n)
    s = _solver(hip, solver="gmres", blockRows=rows, maxIters=1, tolerance=1e-14)
    s.set(A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data)
    s.set_rhs(b)
    o = s.ordering_info()
    assert o == {"blocks": 2 * per_colour, "colours": 2}
    s.solve(raise_on_noconv=False)
    perm, rp, ci, v = s.ilu_export()
    x, r = s.x()[perm], b[perm]
    F = sp.csr_matrix((v, ci, rp), shape=(n, n))
    L, U = sp.tril(F, -1).tocsr() + sp.identity(n, format="csr"), sp.triu(F).tocsr()
    lux = L @ (U @ x)
    alpha = (lux @ r) / (r @ r)
    assert np.all(np.abs(lux - alpha * r) <= 32 * 2.0 ** -53 * (abs(L) @ (abs(U) @ np.abs(x)) + np.abs(alpha * r)))


def test_export_roundtrip(hip, tri_case):
    rp, ci, v, b = tri_case
    s = _solver(hip)
    s.set(rp, ci, v)
    s.set_rhs(b)
    erp, eci, ev, erhs = s.export()
    keep = ci >= 0
    assert np.array_equal(eci, ci[keep])
    assert np.array_equal(ev, v[keep])
    assert np.array_equal(erhs, -b)


@pytest.mark.parametrize("solver", ["bicgstab", "cg"])
@pytest.mark.parametrize("mode", ["fp64", "mixed"])
def test_solve_matches_direct(hip, tri_case, mode, solver):
    """BiCGStab (the reference's default Belos solver) and preconditioned CG
    (Belos "CG", for the symmetric pressure matrix) against a direct solve."""
    rp, ci, v, b = tri_case
    A = H.compact_sorted(rp, ci, v).tocsc()
    x_ref = spla.splu(A).solve(b)
    s = _solver(hip, mode=mode, tolerance=1e-8, maxIters=5000, solver=solver)
    s.set(rp, ci, v)
    s.set_rhs(b)
    rel = s.solve()
    x = s.x()
    true_rel = np.linalg.norm(b - A @ x) / np.linalg.norm(b)
    assert rel <= 1e-8
    assert true_rel <= 1.5e-8
    # ||x - x*|| / ||x*|| <= cond * relres; cond of this system ~1e4..1e5
    assert np.linalg.norm(x - x_ref) / np.linalg.norm(x_ref) <= 1e-3
    st = s.stats()
    assert st["inner_iters"] > 0 and st["solve_ms"] > 0


def test_solve_rectilinear_closed_form(hip, oracle):
    """5-point Poisson with a manufactured solution x* (b = A x*)."""
    xy, cptr, cind = H.rect_case(64, 64)
    m, (rp, ci, v), _, g, bc = H.pressure_system(oracle, xy, cptr, cind, sigma=0.0)
    n = len(rp) - 1
    xs = np.sin(np.arange(n) * 0.37)
    b = oracle.spmv(rp, ci, v, xs)
    for mode in ("fp64", "mixed"):
        s = _solver(hip, mode=mode, tolerance=1e-10, maxIters=4000)
        s.set(rp, ci, v)
        s.set_rhs(b)
        s.solve()
        assert np.linalg.norm(s.x() - xs) / np.linalg.norm(xs) < 1e-6


def test_warm_start_and_guess(hip, tri_case):
    rp, ci, v, b = tri_case
    s = _solver(hip, tolerance=1e-8, maxIters=5000)
    s.set(rp, ci, v)
    s.set_rhs(b)
    s.solve()
    it1 = s.n_iters()
    # same system again: the previous solution is the initial guess
    s.set(rp, ci, v)
    s.set_rhs(b)
    s.solve()
    assert s.n_iters() <= 1 < it1 + 1
    s.set_guess(np.zeros(len(b)))
    s.solve()
    assert s.n_iters() == it1


def test_noconvergence_reported(hip, tri_case):
    rp, ci, v, b = tri_case
    s = _solver(hip, tolerance=1e-12, maxIters=3)
    s.set(rp, ci, v)
    s.set_rhs(b)
    with pytest.raises(hip.PhaseHipError) as ei:
        s.solve()
    assert ei.value.code == -4
    assert s.n_iters() <= 3 + 8


def test_unknown_solver_rejected(hip):
    with pytest.raises(hip.PhaseHipError):
        _solver(hip, solver="tfqmr")


def test_bad_pattern_rejected(hip):
    s = _solver(hip)
    with pytest.raises(hip.PhaseHipError):
        s.set(np.array([0, 1, 2], np.int32), np.array([0, 7], np.int32), np.ones(2))


def test_variable_density_pressure(hip, oracle):
    """The rising-bubble pressure equation, laplacian(dt / rho_f, p) == src::div(u)
    with density ratio 1000 (FractionalStepMultiphase.cpp:152-154), assembled on
    the device: FP64 and mixed both reach the FP64 true residual 1e-8 and agree
    with the oracle's assembly + direct solve."""
    from phase_amd import meshgen as G

    xy, cptr, cind = G.rectilinear(32, 64, width=1.0, height=2.0)
    om = oracle.Mesh(xy, cptr, cind)
    hm = hip.HipMesh(xy, cptr, cind)
    f = om.faces()
    fc = f["centroid"]
    a, b = xy[f["lnode"]], xy[f["rnode"]]
    top = (f["rcell"] < 0) & (a[:, 1] == 2.0) & (b[:, 1] == 2.0)
    bc = np.where(top, hip.BC_FIXED, hip.BC_NORMAL_GRADIENT).astype(np.int32)
    rho = np.where((fc[:, 0] - 0.5) ** 2 + (fc[:, 1] - 0.5) ** 2 < 0.0625, 1.0, 1000.0)
    gamma = 1e-4 / rho
    rhs = G.zero_mean_normal(om.n_cells, seed=7)
    e = oracle.laplacian(om, 3, gamma_face=gamma, bc_type=bc, phi_face=np.zeros(om.n_faces))
    e -= rhs
    rp, ci, v, r = e.get()
    A = H.compact_sorted(rp, ci, v)
    xs = spla.spsolve(A.tocsc(), -r)
    for mode, solver in (("fp64", "bicgstab"), ("mixed", "bicgstab"), ("fp64", "cg"), ("mixed", "cg")):
        s = hip.HipSparseMatrixSolver(0, tolerance=1e-8, maxIters=20000, mode=mode, solver=solver)
        s.assemble_laplacian_device(hm, 3, gamma_face=hip.DeviceArray(gamma), bc_type=hip.DeviceArray(bc),
                                    phi_face=hip.DeviceArray(np.zeros(om.n_faces)))
        s.sub_rhs_device(hip.DeviceArray(rhs))
        rr = s.solve()
        x = s.x()
        assert rr <= 1e-8
        assert np.linalg.norm(-r - A @ x) <= 1.5e-8 * np.linalg.norm(r)
        # the system is ill-conditioned by the density jump: the solution error
        # is bounded by kappa * 1e-8, far looser than the residual
        assert np.linalg.norm(x - xs) <= 1e-3 * np.linalg.norm(xs)


@pytest.mark.parametrize("mode,solver", [("fp64", "bicgstab"), ("mixed", "cg")])
def test_repeated_solves_are_bit_identical(hip, tri_case, mode, solver):
    """Every reduction sums per-block partials in a fixed order, so the same
    solve twice gives the same iterates: identical x bits and iteration
    counts, on one solver and on a fresh one."""
    rp, ci, v, b = tri_case
    out = []
    for fresh in (False, False, True):
        if not out or fresh:
            s = _solver(hip, mode=mode, tolerance=1e-8, maxIters=5000, solver=solver)
            s.set(rp, ci, v)
        s.set_rhs(b)
        s.set_guess(np.zeros(len(b)))
        s.solve()
        out.append((s.x(), s.n_iters(), s.stats()["outer_passes"]))
    for x, it, passes in out[1:]:
        assert np.array_equal(x, out[0][0]) and it == out[0][1] and passes == out[0][2]


def test_mixed_unconverged_finishes_in_fp64(hip, tri_case):
    """A mixed solve that stops above the tolerance with iterations left (here
    forced from the host: no FP32 refinement pass allowed) continues in FP64
    from its best iterate instead of returning unconverged."""
    rp, ci, v, b = tri_case
    A = H.compact_sorted(rp, ci, v)
    for solver in ("bicgstab", "cg"):
        s = _solver(hip, mode="mixed", tolerance=1e-8, maxIters=5000, solver=solver, maxOuter=0)
        s.set(rp, ci, v)
        s.set_rhs(b)
        assert s.solve() <= 1e-8
        assert s.stats()["fallbacks"] == 1
        assert np.linalg.norm(b - A @ s.x()) <= 1.5e-8 * np.linalg.norm(b)
