"""Kernel variants at the sizes where their dispatch changes or their tiles
end: each against the oracle or a sparse LU solve of the same system."""
import numpy as np
import pytest

from test_gpu_mg import _reference
from test_gpu_stokes import _stokes

pytestmark = pytest.mark.gpu

# The one-workgroup coarse end: whole requests of up to 2048 rows (P1 44 / 45,
# P2 22 / 23, elasticity 31 / 32), level sets that do and do not fit LDS (P2 16
# / 17, elasticity 21 / 31), odd and even coarsening, one level only.
COARSE = [(1, 1, 2), (1, 1, 44), (1, 1, 45), (1, 1, 63), (1, 2, 16), (1, 2, 17), (1, 2, 22), (1, 2, 23), (2, 1, 4),
          (2, 1, 21), (2, 1, 31), (2, 1, 32), (2, 1, 48), (2, 1, 49)]


@pytest.mark.parametrize("batch", [0, 16])
def test_coarse_end_matches_lu(grmp, O, batch):
    """1e-8: the residual is 1e-12 and these systems' condition below 1e4"""
    print(f"[case] one-workgroup coarse end, batch {batch}", flush=True)
    with grmp.Server("mg", mg_batch=batch) as S:
        ts = [S.submit(*spec, 40 + k, rtol=1e-12) for k, spec in enumerate(COARSE)]
        for k, (spec, t) in enumerate(zip(COARSE, ts)):
            r = S.wait(t)
            x = _reference(grmp, O, *spec, 40 + k)
            err = np.linalg.norm(S.solution(t) - x) / max(np.linalg.norm(x), 1e-300)
            assert r.status == 0 and r.iterations <= 40 and err <= 1e-8, (spec, r.status, r.iterations, err)


def _fan(k):
    """k triangles around one vertex: its row has k + 1 columns"""
    t = 2.0 * np.pi * np.arange(k) / k
    r = 1.0 + 0.2 * np.cos(3.0 * t)
    coords = np.vstack([[0.03, 0.02], np.column_stack([r * np.cos(t), r * np.sin(t)])])
    cells = np.column_stack([np.zeros(k, int), 1 + np.arange(k), 1 + (np.arange(k) + 1) % k])
    return coords, cells


# row widths at the pattern kernel's set sizes (32, 64, 255 columns)
@pytest.mark.parametrize("width", [4, 31, 32, 33, 64, 65, 200, 255])
def test_pattern_row_widths(grmp, O, width):
    """The pattern is the oracle's exactly, and so are the values."""
    print(f"[case] pattern of a row with {width} columns", flush=True)
    coords, cells = _fan(width - 1)
    grid = grmp.ExtendableGrid.from_arrays(coords, cells)
    fes = grmp.FESpace(grmp.H1P1(1), grid)
    A = grmp.FEMatrix([fes])
    form, keep = grmp.LaplaceOperator(0.7).form(fes, 0, 0, fes.ctx)
    A.add_form(form, keep)
    A.set_fixed(np.array([1, 3]))
    A.build_pattern()
    A.assemble()
    cp, rv, nz = A.csc()
    ref = O.assemble_matrix(fes.ndofs, [dict(kind=O.BLF_LAPLACE, fe=O.FE_P1, quadorder=0, factor=0.7, coords=coords,
                                             cells=cells, celldofs=cells)], fixed=np.array([1, 3]))
    assert A.info()[2] == width
    assert np.array_equal(cp, ref.colptr) and np.array_equal(rv, ref.rowval) and np.array_equal(nz, ref.nzval)


def test_pattern_row_too_wide(grmp):
    print("[case] pattern of a row with 256 columns", flush=True)
    coords, cells = _fan(255)
    grid = grmp.ExtendableGrid.from_arrays(coords, cells)
    fes = grmp.FESpace(grmp.H1P1(1), grid)
    A = grmp.FEMatrix([fes])
    form, keep = grmp.LaplaceOperator(1.0).form(fes, 0, 0, fes.ctx)
    A.add_form(form, keep)
    with pytest.raises(grmp.GrmpError) as e:
        A.build_pattern()
    assert e.value.code == grmp._abi.ERR_UNSUPPORTED


# coarse rows of the Galerkin product at its set sizes: aggregated pairs halve
# a hub's columns (24 and 42 of 48 and 84, 125 of 250); three hubs in one
# aggregate have about 376, more than a set holds
@pytest.mark.parametrize("hubs,k", [(1, 48), (1, 84), (1, 250), (3, 250)])
def test_amg_wide_coarse_rows(grmp, hubs, k):
    """1e-8 against LU: the residual is 1e-12, the condition below 1e4"""
    print(f"[case] algebraic multigrid, {hubs} hub(s) of {k} cells", flush=True)
    import scipy.sparse.linalg as spla
    co, ce = [], []
    for h in range(hubs):
        c, e = _fan(k)
        t = 2.0 * np.pi * h / 3.0
        co.append(c + 5.0 * np.array([np.cos(t), np.sin(t)]))
        ce.append(e + h * (k + 1))
    if hubs == 3:
        ce.append(np.array([[0, k + 1, 2 * (k + 1)]]))
    grid = grmp.ExtendableGrid.from_arrays(np.vstack(co), np.vstack(ce))
    fes = grmp.FESpace(grmp.H1P1(1), grid)
    pde = grmp.PoissonProblem(1.0)
    pde.add_operator((0, 0), grmp.ReactionOperator(0.01))
    pde.add_rhsdata(0, grmp.LinearForm(grmp.Identity, grmp.DataFunction([1.0])))
    pde.add_rhsdata(0, grmp.LinearForm(grmp.Identity, grmp.PolynomialData([0.0, 1.0, -0.5])))
    sol = grmp.FEVector([fes])
    info, A, b = grmp.solve(sol, pde, solver="amg", rtol=1e-12)
    x = spla.spsolve(A.to_scipy().tocsc(), b.entries())
    err = np.linalg.norm(sol.entries() - x) / np.linalg.norm(x)
    assert info.status == 0 and err <= 1e-8, (info.iterations, err)


# plain CG: two launches an iteration up to 512 workgroups of 256 rows, five
# beyond (P1 361 x 361 nodes: 130,321 rows, 510 workgroups; 363 x 363: 515);
# FP32 sweeps: tiles of one problem alone
@pytest.mark.parametrize("precision", ["fp64", "fp32_ir"])
@pytest.mark.parametrize("N", [1, 2, 15, 16, 63, 360, 362])
def test_krylov_cg_sizes(grmp, O, N, precision):
    """1e-8 against LU: the residual is 1e-12, the condition of these systems
    at most 1e5"""
    print(f"[case] Jacobi CG, P1 {N}x{N}, {precision}", flush=True)
    grid = grmp.grid_unitsquare(N)
    fes = grmp.FESpace(grmp.H1P1(1), grid)
    pde = grmp.PoissonProblem(1.0)
    pde.add_rhsdata(0, grmp.LinearForm(grmp.Identity, grmp.DataFunction([1.0])))
    pde.add_boundarydata(0)
    sol = grmp.FEVector([fes])
    info, A, b = grmp.solve(sol, pde, precision=precision, rtol=1e-12)
    import scipy.sparse.linalg as spla
    x = spla.spsolve(A.to_scipy().tocsc(), b.entries())
    err = np.linalg.norm(sol.entries() - x) / max(np.linalg.norm(x), 1e-300)
    assert info.status == 0 and err <= 1e-8, (info.iterations, err)


def test_krylov_cg_iteration_cap(grmp):
    """The cap and a start at the solution end both forms as before."""
    print("[case] Jacobi CG, iteration cap", flush=True)
    for N in (40, 400):
        grid = grmp.grid_unitsquare(N)
        fes = grmp.FESpace(grmp.H1P1(1), grid)
        pde = grmp.PoissonProblem(1.0)
        pde.add_rhsdata(0, grmp.LinearForm(grmp.Identity, grmp.DataFunction([1.0])))
        pde.add_boundarydata(0)
        sol = grmp.FEVector([fes])
        with pytest.raises(grmp.GrmpError) as e:
            grmp.solve(sol, pde, rtol=1e-12, maxiterations=5)
        assert e.value.code == grmp._abi.ERR_NOCONV and "after 5 iterations" in str(e.value)
        pde0 = grmp.PoissonProblem(1.0)
        pde0.add_boundarydata(0)
        info, A, b = grmp.solve(grmp.FEVector([fes]), pde0, rtol=1e-12)
        assert info.status == 0 and info.iterations == 0


# The levels' FP32 values and bounds: rows in whole blocks of 256 (P1 15, 31
# and 127, elasticity 63) and just past them (P1 16), more than 2048 nonzeros
# in a block (P2, elasticity)
@pytest.mark.parametrize("spec", [(1, 1, 15), (1, 1, 16), (1, 1, 31), (1, 1, 127), (1, 2, 15), (1, 2, 63), (2, 1, 63)])
def test_level_setup_matches_lu(grmp, O, spec):
    """1e-8: the residual is 1e-12 and these systems' condition below 1e4; a
    wrong value or bound shows in the iterations"""
    print(f"[case] level setup {spec}", flush=True)
    with grmp.Server("mg", mg_block_rows=64) as S:
        t = S.submit(*spec, 7, rtol=1e-12)
        r = S.wait(t)
        x = _reference(grmp, O, *spec, 7)
        err = np.linalg.norm(S.solution(t) - x) / np.linalg.norm(x)
        assert r.status == 0 and r.iterations <= 60 and err <= 1e-8, (r.status, r.iterations, err)


# the fused residual and restriction up to 32,768 rows (P1 180^2 has 32,761),
# two launches beyond; constant coefficients on generated squares
@pytest.mark.parametrize("N", [20, 180, 181])
def test_amg_resid_restrict_sizes(grmp, O, N):
    """3e-8 against LU: the residual is 1e-12, the condition below 4/pi^2 N^2
    8/3 < 3.6e4"""
    print(f"[case] algebraic multigrid, P1 {N}x{N}", flush=True)
    import scipy.sparse.linalg as spla
    fes = grmp.FESpace(grmp.H1P1(1), grmp.grid_unitsquare(N))
    pde = grmp.PoissonProblem(1.0)
    pde.add_rhsdata(0, grmp.LinearForm(grmp.Identity, grmp.DataFunction([1.0])))
    pde.add_boundarydata(0)
    sol = grmp.FEVector([fes])
    info, A, b = grmp.solve(sol, pde, solver="amg", rtol=1e-12)
    x = spla.spsolve(A.to_scipy().tocsc(), b.entries())
    err = np.linalg.norm(sol.entries() - x) / np.linalg.norm(x)
    assert info.status == 0 and err <= 3e-8, (info.iterations, err)


# 256 rows' columns are put together in LDS up to 6144 of them: hubs numbered
# first, 21 (5355 and 235 rim rows of 4 are 6295) and 64 do not fit, 4 do; the
# rim rows' blocks do
@pytest.mark.parametrize("hubs,k", [(4, 254), (21, 254), (64, 254)])
def test_pattern_columns_in_place(grmp, O, hubs, k):
    """The pattern and values are the oracle's bit for bit."""
    print(f"[case] pattern of {hubs} hubs of {k} cells", flush=True)
    c0, e0 = _fan(k)
    coords = np.vstack([c0[:1] + [5.0 * h, 0.0] for h in range(hubs)] +
                       [c0[1:] + [5.0 * h, 0.0] for h in range(hubs)])
    cells = np.vstack([np.where(e0 == 0, h, hubs + h * k + e0 - 1) for h in range(hubs)])
    grid = grmp.ExtendableGrid.from_arrays(coords, cells)
    fes = grmp.FESpace(grmp.H1P1(1), grid)
    A = grmp.FEMatrix([fes])
    form, keep = grmp.LaplaceOperator(0.7).form(fes, 0, 0, fes.ctx)
    A.add_form(form, keep)
    A.build_pattern()
    A.assemble()
    cp, rv, nz = A.csc()
    ref = O.assemble_matrix(fes.ndofs, [dict(kind=O.BLF_LAPLACE, fe=O.FE_P1, quadorder=0, factor=0.7, coords=coords,
                                             cells=cells, celldofs=cells)])
    assert np.array_equal(cp, ref.colptr) and np.array_equal(rv, ref.rowval) and np.array_equal(nz, ref.nzval)


# whole and partial blocks of 256 rows, and 1 to 24 incidences a dof, in fours
# and not
@pytest.mark.parametrize("n", [1, 2, 5, 6, 7])
def test_tet_pattern_and_load_sizes(grmp, O, n):
    """Pattern, values and load vector are the oracle's bit for bit."""
    print(f"[case] tetrahedra n={n}", flush=True)
    grid = grmp.grid_unitcube(n, 0.1, n)
    c, cn = grid.download()
    fes = grmp.FESpace(grmp.H1P1(1), grid)
    A = grmp.FEMatrix([fes])
    form, keep = grmp.LaplaceOperator(0.7).form(fes, 0, 0, fes.ctx)
    A.add_form(form, keep)
    A.build_pattern()
    A.assemble()
    cp, rv, nz = A.csc()
    ref = O.assemble_matrix(fes.ndofs, [dict(kind=O.BLF_LAPLACE, geom=3, fe=O.FE_P1, quadorder=0, factor=0.7, coords=c,
                                             cells=cn, celldofs=cn)])
    assert np.array_equal(cp, ref.colptr) and np.array_equal(rv, ref.rowval) and np.array_equal(nz, ref.nzval)
    b = grmp.FEVector([fes])
    grmp.assemble_linearform(b, 0, grmp.LinearForm(grmp.Identity, grmp.DataFunction([1.5])))
    bref = np.zeros(fes.ndofs)
    O.assemble_lf_const(bref, O.FE_P1, 1, 1, [1.5], c, cn, cn, geom=3)
    assert np.array_equal(b.entries(), bref)


# Group setup: one request, a whole group and one more; single-level requests,
# whole 256-row blocks and one row past them, levels in and out of LDS
@pytest.mark.parametrize("count", [1, 16, 17])
def test_group_setup_equals_alone(grmp, count):
    """The same bits as each request set up and solved by itself.  The one setup
    thread is at work on a large request while the others come, so it takes them
    in groups of 16: all were there before the first was begun."""
    print(f"[case] setup of {count} requests", flush=True)
    shapes = [(1, 1, 15), (1, 2, 33), (2, 1, 3), (1, 1, 2), (2, 1, 63), (1, 1, 16), (1, 2, 2), (1, 1, 127)]
    reqs = [(*shapes[k % len(shapes)], 60 + k) for k in range(count)]
    out = []
    for kw in ({"mg_slots": 1, "mg_batch": 0}, {"mg_batch": 32, "mg_threads": 1}):
        with grmp.Server("mg", mg_block_rows=1000, mg_coarse_rows=1000, **kw) as S:
            S.submit(1, 2, 500, 59, keep_solution=False)
            ts = [S.submit(*r, rtol=1e-11) for r in reqs]
            res = [S.wait(t) for t in ts]
            out.append([(r.iterations, S.solution(t).copy()) for r, t in zip(res, ts)])
            if kw["mg_batch"]:
                assert max(r.t_submit for r in res) < min(r.t_admit for r in res)
    for r, (ia, xa), (ib, xb) in zip(reqs, *out):
        assert ia == ib and np.array_equal(xa, xb), r


# rtol below the floor of b - A x: the check in the batch asks for restarts,
# up to three, and accepts within 100 rtol
@pytest.mark.parametrize("rtol", [1e-14, 3e-15])
def test_batch_restarts_equal_alone(grmp, rtol):
    """The same bits, iterations and status as each request by itself"""
    print(f"[case] restarts in a batch, rtol {rtol}", flush=True)
    reqs = [(1, 1, 65, 3), (1, 2, 48, 4), (2, 1, 40, 5), (1, 1, 120, 6), (1, 1, 9, 7)]
    out = []
    for kw in ({"mg_slots": 1, "mg_batch": 0}, {"mg_batch": 8}, {"mg_batch": 8, "mg_threads": -1}):
        with grmp.Server("mg", mg_block_rows=256, mg_coarse_rows=256, **kw) as S:
            ts = [S.submit(*r, rtol=rtol) for r in reqs]
            res = [S.wait(t) for t in ts]
            out.append([(r.status, r.iterations, r.relres, S.solution(t).copy()) for r, t in zip(res, ts)])
    assert any(o[2] > rtol for o in out[0])  # at least one was checked and restarted
    for got in out[1:]:
        for r, a, b in zip(reqs, out[0], got):
            assert a[:3] == b[:3] and np.array_equal(a[3], b[3]), (r, a[:3], b[:3])


def _bicgstab(grmp, A, b, maxit, pc=None, rtol=1e-13):
    """(status, iterations, relres, x) of BiCGStab stopped after maxit steps"""
    import ctypes
    o, info = grmp._abi.SolveOpts(), grmp._abi.SolveInfo()
    L = grmp.lib()
    L.grmp_solve_opts_default(ctypes.byref(o))
    o.method, o.precision, o.rtol, o.maxit = grmp._abi.SOLVE_BICGSTAB, grmp._abi.PRECISION_FP64, rtol, maxit
    x = grmp.DeviceVector(A.ctx, A.n)
    if pc:
        rc = L.grmp_solve_bicgstab_amg(A.h, b.h, x.h, ctypes.byref(o), pc.h, ctypes.byref(info))
    else:
        rc = L.grmp_solve(A.h, b.h, x.h, ctypes.byref(o), ctypes.byref(info))
    assert rc == info.status
    return info.status, info.iterations, info.relres, x.download()


def _newton_matrix(grmp, n=9):
    """A P2 Newton matrix (nonsymmetric) with its boundary fixed, a right-hand
    side, and both on the host"""
    fes = grmp.FESpace(grmp.H1P2(1), grmp.grid_unitsquare(n))
    nlf = grmp.NonlinearForm(grmp.Gradient, [grmp.Identity, grmp.Gradient], [0, 0],
                             grmp.NonlinearDiffusion(1.0, 0.0, 1.0), [2, 3], bonus_quadorder=2)
    X = grmp.FEVector([fes])
    X.set_entries(np.random.default_rng(3).standard_normal(fes.ndofs))
    A = grmp.FEMatrix([fes])
    A.add_form(*nlf.form(fes, 0, 0, fes.ctx, current=X))
    A.set_fixed(fes.boundary_dofs())
    A.assemble(grmp._abi.VALUES_FP64)
    bh = np.random.default_rng(4).standard_normal(fes.ndofs)
    b = grmp.DeviceVector(fes.ctx, fes.ndofs)
    b.upload(bh)
    free = np.ones(fes.ndofs, bool)
    free[fes.boundary_dofs()] = False
    return A, b, A.to_scipy().tocsr(), bh, free


def _bicgstab_host(K, b, free, steps):
    """x and |r| / |r_0| after steps of right-Jacobi BiCGStab on the free rows"""
    d = K.diagonal()
    x = np.where(free, 0.0, b / d)
    mul = lambda v: np.where(free, K @ v, 0.0)
    dinv = np.where(free, 1.0 / d, 0.0)
    r = np.where(free, b - K @ x, 0.0)
    rh, p, rho, r0 = r.copy(), r.copy(), r @ r, np.linalg.norm(r)
    for _ in range(steps):
        ph = dinv * p
        v = mul(ph)
        alpha = rho / (rh @ v)
        s = r - alpha * v
        sh = dinv * s
        t = mul(sh)
        omega = (s @ t) / (t @ t)
        x = x + alpha * ph + omega * sh
        r = s - omega * t
        rho, old = rh @ r, rho
        p = r + (rho / old) * (alpha / omega) * (p - omega * v)
    return x, np.linalg.norm(r) / r0


# BiCGStab's steps are enqueued two at a time: caps inside a pair and at its end
@pytest.mark.parametrize("maxit", [1, 2, 3, 5])
def test_bicgstab_iteration_cap(grmp, maxit):
    """Exactly maxit steps, x and the residual those of the recurrence on the
    host: 1e-12 (on the host, five steps in 64 and in 80 bits differ by 4e-16).
    With a V-cycle the residual is that of the x returned: nothing enqueued
    behind the last step touches it."""
    print(f"[case] BiCGStab stopped after {maxit} steps", flush=True)
    A, b, K, bh, free = _newton_matrix(grmp)
    xh, relh = _bicgstab_host(K, bh, free, maxit)
    st, it, rel, x = _bicgstab(grmp, A, b, maxit)
    assert st == grmp._abi.ERR_NOCONV and it == maxit
    assert np.linalg.norm(x - xh) <= 1e-12 * np.linalg.norm(xh) and abs(rel - relh) <= 1e-12, (rel, relh)
    x0 = np.where(free, 0.0, bh / K.diagonal())
    r0 = np.linalg.norm((bh - K @ x0)[free])
    for pc in (None, grmp.AlgebraicMultigridSolver(A)):
        st, it, rel, x = _bicgstab(grmp, A, b, maxit, pc)
        true = np.linalg.norm((bh - K @ x)[free]) / r0
        assert st == grmp._abi.ERR_NOCONV and it == maxit and abs(rel - true) <= 1e-12, (pc, rel, true)


def test_bicgstab_ends(grmp):
    """A right-hand side with a NaN ends at once; one free row converges in the
    first half of a step (s = 0)."""
    print("[case] BiCGStab ends", flush=True)
    A, b, K, bh, free = _newton_matrix(grmp, 5)
    bh[np.flatnonzero(free)[3]] = np.nan
    b.upload(bh)
    for pc in (None, grmp.AlgebraicMultigridSolver(A)):
        st, it, rel, x = _bicgstab(grmp, A, b, 50, pc)
        assert st == grmp._abi.ERR_NONFINITE and it == 0, (pc, st, it)
    fes = grmp.FESpace(grmp.H1P1(1), grmp.grid_unitsquare(2))
    A = grmp.FEMatrix([fes])
    A.add_form(*grmp.LaplaceOperator(1.0).form(fes, 0, 0, fes.ctx))
    A.set_fixed(fes.boundary_dofs())
    A.assemble(grmp._abi.VALUES_FP64)
    b = grmp.DeviceVector(fes.ctx, fes.ndofs)
    b.upload(np.where(np.arange(fes.ndofs) == 4, 3.0, 0.0))
    st, it, rel, x = _bicgstab(grmp, A, b, 50)
    assert st == 0 and it == 1 and rel == 0.0 and np.array_equal(x, np.where(np.arange(9) == 4, 0.75, 0.0))


# the whole hierarchy in one workgroup (P1 16^2) and grid levels over it (64^2)
@pytest.mark.parametrize("N", [16, 64])
def test_hierarchy_for_cg_and_minres_in_turn(grmp, N):
    """CG takes the smoother's coefficients of the fourth kind, MINRES of the
    first: each use gives the same bits before and after the other."""
    print(f"[case] one hierarchy under CG, MINRES and CG, {N}x{N}", flush=True)
    grid, V, Q, pde, sol = _stokes(grmp, N)
    A, b, fixed = grmp.assemble(pde, sol)
    M = grmp.stokes_velocity_mg(pde, V)
    cfg = grmp.SolverConfig(rtol=1e-9)
    f = grmp.FEVector([M.levels[0][1]])
    f.set_entries(np.random.default_rng(N).standard_normal(f.n))

    def cg():
        x = grmp.FEVector([M.levels[0][1]])
        info = M.solve(f, x, 1e-10)
        return info.iterations, x.entries()

    def minres():
        info = grmp.solve_system(A, b, sol, cfg, grmp._abi.SOLVE_MINRES, velocity_mg=M)
        return info.iterations, sol.entries().copy()

    first, second = (cg(), minres()), (cg(), minres())
    for (ia, xa), (ib, xb) in zip(first, second):
        assert ia == ib and np.array_equal(xa, xb), (ia, ib)


@pytest.mark.parametrize("N", [30, 200])
def test_fourth_kind_goes_on_below_rtol(grmp, N):
    """P1 hierarchies under CG stop at 0.4 rtol (the error at a given residual is
    larger with their smoother); at the cap rtol itself is enough."""
    print(f"[case] margin below rtol, P1 {N}x{N}", flush=True)
    fes = grmp.FESpace(grmp.H1P1(1), grmp.grid_unitsquare(N))
    pde = grmp.PoissonProblem(1.0)
    pde.add_rhsdata(0, grmp.LinearForm(grmp.Identity, grmp.DataFunction([1.0])))
    pde.add_boundarydata(0)
    sol = grmp.FEVector([fes])
    A, b, fixed = grmp.assemble(pde, sol)
    M = grmp.MultigridSolver(*grmp.mg_hierarchy(pde, fes, A))
    i0 = M.solve(b, sol, 1e-8)
    assert i0.status == 0 and i0.relres <= 0.4e-8
    rtol = 1.5 * i0.relres  # met by the residual of i0, its margin is not
    i1 = M.solve(b, sol, rtol)
    assert i1.status == 0 and i1.iterations == i0.iterations + 1 and i1.relres <= 0.4 * rtol
    i2 = M.solve(b, sol, rtol, maxit=i0.iterations)
    assert i2.status == 0 and i2.iterations == i0.iterations and i2.relres <= rtol
    with pytest.raises(grmp.GrmpError) as e:
        M.solve(b, sol, rtol, maxit=i0.iterations - 1)
    assert e.value.code == grmp._abi.ERR_NOCONV
