"""Kernel variants at the sizes where their dispatch changes or their tiles
end: each against the oracle or a sparse LU solve of the same system."""
import numpy as np
import pytest

from test_gpu_mg import _reference

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
    """The same bits as each request set up and solved by itself"""
    print(f"[case] setup of {count} requests", flush=True)
    shapes = [(1, 1, 15), (1, 2, 33), (2, 1, 3), (1, 1, 2), (2, 1, 63), (1, 1, 16), (1, 2, 2), (1, 1, 127)]
    reqs = [(*shapes[k % len(shapes)], 60 + k) for k in range(count)]
    out = []
    for kw in ({"mg_slots": 1, "mg_batch": 0}, {"mg_batch": 32, "mg_threads": 1}):
        with grmp.Server("mg", mg_block_rows=1000, mg_coarse_rows=1000, **kw) as S:
            ts = [S.submit(*r, rtol=1e-11) for r in reqs]
            out.append([(S.wait(t).iterations, S.solution(t).copy()) for t in ts])
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
