"""Timed cases of the assembly-and-solve engine, from the calls its users make.

Every case goes through the package's public entry points (``solve``,
``FEMatrix.assemble``, ``TimeControlSolver.advance``, ``Server.submit`` ...) on
the workloads and size ranges of the repository's own configurations: 2D
Poisson and elasticity with log-normal cell coefficients on squares of up to
2048 x 2048, jittered tetrahedral cubes of up to 160^3, gradient-robust Stokes
on up to 512 x 512, the heat equation, the nonlinear Poisson equation, uploaded
meshes, and the served request stream.

``listed`` gives the fixed cases, ``draw`` another one of the same ranges,
``prepare`` what a program holds before the call (grid, coefficient, problem),
``run`` one pass, ``work`` the bytes and operations no implementation can avoid,
``tolerance`` what correct implementations of the same precision differ by, and
``exact`` the outputs from plain torch in 64 bits.
"""
import math
import random

import numpy as np
import torch

import __graft_entry__ as _entry

grmp = _entry.load()
_abi = grmp._abi

# relative residual of the solves: the single-instance configurations' 1e-10,
# the served stream's 1e-9, the Newton loop's inner 1e-12
RTOL, RTOL_SERVED, RTOL_NEWTON = 1e-10, 1e-9, 1e-12
# the Newton loop's own target: the residual's rounding floor is below 1e-9 over
# these sizes and data, and the sixth step reaches it
RESIDUAL_NEWTON = 5e-9


def listed():
    return [
        # the plain method on the small configuration, default solver (Jacobi CG): launches and latency count
        dict(name="solve-p2-64-krylov", kind="solve", pde="poisson", fe=2, n=64, coef=False, solver="krylov",
             precision="fp64"),
        # elasticity as an ordinary call, the solver chosen by the library (geometric multigrid), odd size
        dict(name="solve-elasticity-383", kind="solve", pde="elasticity", fe=1, n=383, coef=True, solver="auto",
             precision="fp64"),
        # P2 at the size of the large 2D configuration (4.2M dofs), odd
        dict(name="solve-p2-1023", kind="solve", pde="poisson", fe=2, n=1023, coef=True, solver="auto",
             precision="fp64"),
        # a 3D problem solved from the mesh on: pattern, assembly, algebraic multigrid hierarchy, CG
        dict(name="solve-tet-128", kind="solve", pde="poisson", fe=3, n=128, coef=True, solver="auto",
             precision="fp64"),
        # FP32 sweeps inside FP64 refinement, where that precision option pays (3D)
        dict(name="solve-tet-75-fp32", kind="solve", pde="poisson", fe=3, n=75, coef=True, solver="krylov",
             precision="fp32_ir"),
        # the caller's own triangle mesh, from host arrays: faces, dofmap, interpolated boundary data, solve
        dict(name="upload-p2-211", kind="upload", fe=2, n=211),
        # a new coefficient on a kept pattern: reassembly and one product (a residual), P2 and tetrahedra
        dict(name="assemble-p2-1501", kind="assemble", pde="poisson", fe=2, n=1501),
        dict(name="assemble-tet-160", kind="assemble", pde="poisson", fe=3, n=160),
        # gradient-robust Stokes, the full-size configuration
        dict(name="stokes-512", kind="stokes", n=512),
        # one step of the heat equation on the 2048^2 grid (fixed step size, the system kept)
        dict(name="heat-2048", kind="heat", n=2048),
        # a whole Newton loop of the nonlinear Poisson equation
        dict(name="newton-p2-256", kind="newton", fe=2, n=256),
        # a burst of the served stream: Poisson P1 / P2 and elasticity requests of log-uniform sizes
        dict(name="serve-48", kind="serve", count=48, mix=11),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve2d", "solve2d", "solve2d", "solve3d", "krylov", "fp32", "upload", "assemble", "assemble",
                       "stokes", "heat", "newton", "serve"])
    if kind == "solve2d":
        pde, fe, hi = rng.choice([("poisson", 1, 2048), ("poisson", 2, 1023), ("elasticity", 1, 1023)])
        return dict(kind="solve", pde=pde, fe=fe, n=_log_int(rng, 32, hi), coef=True, solver="auto", precision="fp64")
    if kind == "solve3d":
        return dict(kind="solve", pde="poisson", fe=3, n=_log_int(rng, 12, 128), coef=True, solver="auto",
                    precision="fp64")
    if kind == "krylov":
        pde, fe = rng.choice([("poisson", 1), ("poisson", 2), ("elasticity", 1), ("poisson", 3)])
        return dict(kind="solve", pde=pde, fe=fe, n=_log_int(rng, 16, 48 if fe == 3 else 160), coef=rng.random() < 0.5,
                    solver="krylov", precision="fp64")
    if kind == "fp32":
        return dict(kind="solve", pde="poisson", fe=3, n=_log_int(rng, 12, 96), coef=True, solver="krylov",
                    precision="fp32_ir")
    if kind == "upload":
        return dict(kind="upload", fe=rng.choice([1, 2]), n=_log_int(rng, 24, 320))
    if kind == "assemble":
        pde, fe, hi = rng.choice([("poisson", 1, 2048), ("poisson", 2, 1501), ("poisson", 3, 160),
                                  ("elasticity", 1, 1023)])
        return dict(kind="assemble", pde=pde, fe=fe, n=_log_int(rng, 16 if fe == 3 else 48, hi))
    if kind == "stokes":
        return dict(kind="stokes", n=_log_int(rng, 32, 512))
    if kind == "heat":
        return dict(kind="heat", n=_log_int(rng, 48, 2048))
    if kind == "newton":
        return dict(kind="newton", fe=rng.choice([1, 2]), n=_log_int(rng, 24, 256))
    return dict(kind="serve", count=_log_int(rng, 4, 48), mix=rng.randrange(1 << 20))


# ------------------------------------------------------------------ inputs
def _grid(case, seed):
    if case.get("fe") == 3:
        return grmp.grid_unitcube(case["n"], jitter=0.1, seed=seed)
    return grmp.grid_unitsquare(case["n"])


def _element(case):
    ncomp = 2 if case.get("pde") == "elasticity" else 1
    return grmp.H1P2(ncomp) if case["fe"] == 2 else grmp.H1P1(ncomp)


def _kappa(case, seed, ncells):
    """the log-normal cell coefficient (sigma 1 in 2D, 0.5 in 3D)"""
    kap = grmp.DeviceVector(grmp.default_context(), ncells)
    kap.lognormal(1000003 * seed + 17, 0.0, 0.5 if case.get("fe") == 3 else 1.0)
    return kap


def _problem(case, kap):
    coef = grmp.CellCoefficient(kap) if kap is not None else None
    if case.get("pde") == "elasticity":
        pde = grmp.LinearElasticityProblem(1.0, 0.3, cell_coefficient=coef)
        rhs = [0.0, -1.0]
    else:
        pde = grmp.PoissonProblem(1e-3, cell_coefficient=coef)
        rhs = [1.0]
    return pde, rhs


def _scale(seed):
    """size of the constant right-hand side: 1 up to a seeded factor"""
    return 1.0 + 0.5 * random.Random(seed).random()


def _triangle_mesh(n, seed):
    """A caller's mesh: the n x n triangulated square with its interior nodes
    moved by up to 0.2 h and its cells in a shuffled order."""
    rng = np.random.default_rng(seed)
    g = np.arange(n + 1) / n
    X, Y = np.meshgrid(g, g)
    co = np.column_stack([X.ravel(), Y.ravel()])
    inner = (co > 0).all(1) & (co < 1).all(1)
    co[inner] += rng.uniform(-0.2 / n, 0.2 / n, (int(inner.sum()), 2))
    j, i = np.divmod(np.arange(n * n), n)
    v = j * (n + 1) + i
    cells = np.concatenate([np.column_stack([v, v + 1, v + n + 2]), np.column_stack([v, v + n + 2, v + n + 1])])
    return co, cells[rng.permutation(len(cells))].astype(np.int32)


def _quadratic(seed):
    """coefficients of 1, x, y, x^2, xy, y^2"""
    return np.random.default_rng(seed + 5).uniform(-1.0, 1.0, 6)


def _bilinear(seed):
    """a + b x + c y + d xy: the nonlinear problem's exact solution"""
    return np.random.default_rng(seed + 6).uniform(0.4, 1.0, 4)


def _newton_rhs(c):
    """f = -div((1 + u^2) grad u) = -2 u |grad u|^2 for u = a + b x + c y + d xy,
    as coefficients of the monomials up to degree 4"""
    a, b, cc, d = c
    u = {(0, 0): a, (1, 0): b, (0, 1): cc, (1, 1): d}
    g2 = {}
    for g in ({(0, 0): b, (0, 1): d}, {(0, 0): cc, (1, 0): d}):
        for (i, j), p in g.items():
            for (k, l), q in g.items():
                g2[i + k, j + l] = g2.get((i + k, j + l), 0.0) + p * q
    f = {}
    for (i, j), p in u.items():
        for (k, l), q in g2.items():
            f[i + k, j + l] = f.get((i + k, j + l), 0.0) - 2.0 * p * q
    return [f.get(m, 0.0) for m in grmp.PolynomialData.MONOMIALS]


def _requests(case):
    """The burst's requests, drawn as the benchmark draws its stream; the sizes
    belong to the case, the coefficients to the seed."""
    r = random.Random(case["mix"])
    out = []
    for _ in range(case["count"]):
        kind = r.choice([1, 2])
        out.append((kind, r.choice([1, 2]) if kind == 1 else 1, _log_int(r, 16, 768)))
    return out


def _request_seed(seed, k):
    return 7919 * seed + 104729 * k + 1


def _initial_heat(n, seed):
    a = np.random.default_rng(seed + 9).uniform(0.5, 1.5, 4)
    g = np.arange(n + 1) / n
    X, Y = np.meshgrid(g, g)
    u = sum(a[k] * np.sin((k + 1) * np.pi * X) * np.sin((4 - k) * np.pi * Y) for k in range(4))
    return np.ascontiguousarray(u.ravel())


HEAT_DT = 1e-4


class _Result(np.ndarray):
    """an array over page-locked memory that keeps its buffer alive"""


def _pinned(ctx, sizes):
    """result arrays of these sizes in one page-locked buffer"""
    buf = _abi.PinnedBuffer(ctx, sum(sizes))
    out, off = [], 0
    for m in sizes:
        v = buf.view(off, m).view(_Result)
        v.buffer = buf
        out.append(v)
        off += m
    return out


def prepare(case, seed):
    kind = case["kind"]
    ctx = grmp.default_context()
    st = dict(case=case, ctx=ctx)
    if kind == "solve":
        grid = _grid(case, seed)
        kap = _kappa(case, seed, grid.ncells) if case["coef"] else None
        pde, rhs = _problem(case, kap)
        pde.add_rhsdata(0, grmp.LinearForm(grmp.Identity, grmp.DataFunction([_scale(seed) * v for v in rhs])))
        pde.add_boundarydata(0)
        st.update(grid=grid, fes=grmp.FESpace(_element(case), grid), pde=pde)
    elif kind == "upload":
        co, cells = _triangle_mesh(case["n"], seed)
        kap = np.exp(0.5 * np.random.default_rng(seed + 3).standard_normal(len(cells)))
        st.update(coords=co, cells=cells, kap=kap, data=_quadratic(seed))
    elif kind == "assemble":
        grid = _grid(case, seed)
        kap = _kappa(case, seed, grid.ncells)
        fes = grmp.FESpace(_element(case), grid)
        pde, _ = _problem(case, kap)
        A = grmp.FEMatrix([fes])
        form, keep = pde.LHS[(0, 0)][0].form(fes, 0, 0, ctx)
        A.add_form(form, keep)
        A.build_pattern()
        x = grmp.DeviceVector(ctx, fes.ndofs)
        x.lognormal(seed + 29, 0.0, 1.0)
        st.update(grid=grid, fes=fes, A=A, x=x, y=grmp.DeviceVector(ctx, fes.ndofs),
                  out=_pinned(ctx, [fes.ndofs])[0])
    elif kind == "stokes":
        grid = grmp.grid_unitsquare(case["n"])
        V, Q = grmp.FESpace(grmp.H1BR(2), grid), grmp.FESpace(grmp.L2P0(1), grid)
        rng = np.random.default_rng(seed)
        K = 8
        modes = np.column_stack([rng.normal(0, 0.3, 2 * K), rng.integers(-3, 4, 2 * K), rng.integers(-3, 4, 2 * K),
                                 rng.uniform(0, 2 * np.pi, 2 * K)])
        f = grmp.GradientCurlData(modes[:K], modes[K:], (0.5, -0.25, 0.3), bonus_quadorder=2)
        pde = grmp.IncompressibleNavierStokesProblem(2, viscosity=1e-2)
        pde.add_rhsdata(0, grmp.LinearForm(grmp.ReconstructionIdentity(grmp.HDIVRT0), f))
        st.update(grid=grid, spaces=[V, Q], pde=pde)
    elif kind == "heat":
        grid = grmp.grid_unitsquare(case["n"])
        fes = grmp.FESpace(grmp.H1P1(1), grid)
        pde = grmp.PoissonProblem(cell_coefficient=grmp.CellCoefficient(_kappa(case, seed, grid.ncells)))
        pde.add_rhsdata(0, grmp.LinearForm(grmp.Identity, grmp.DataFunction([1.0])))
        pde.add_boundarydata(0)
        X = grmp.FEVector(fes)
        X.set_entries(_initial_heat(case["n"], seed))
        tcs = grmp.TimeControlSolver(pde, X, grmp.BackwardEuler, timedependent_equations=[0], rtol=RTOL)
        st.update(grid=grid, fes=fes, X=X, tcs=tcs, out=_pinned(ctx, [fes.ndofs])[0])
    elif kind == "newton":
        grid = grmp.grid_unitsquare(case["n"])
        c = _bilinear(seed)
        pde = grmp.PDEDescription("nonlinear Poisson problem")
        pde.add_unknown("u")
        pde.add_operator((0, 0), grmp.NonlinearForm(grmp.Gradient, [grmp.Identity, grmp.Gradient], [0, 0],
                                                    grmp.NonlinearDiffusion(1.0, 0.0, 1.0), [2, 3], bonus_quadorder=2))
        pde.add_boundarydata(0, grmp.InterpolateDirichletBoundary,
                             data=grmp.PolynomialData([c[0], c[1], c[2], 0.0, c[3]]))
        pde.add_rhsdata(0, grmp.LinearForm(grmp.Identity, grmp.PolynomialData(_newton_rhs(c))))
        st.update(grid=grid, fes=grmp.FESpace(_element(case), grid), pde=pde)
    else:
        reqs = _requests(case)
        st.update(reqs=[r + (_request_seed(seed, k),) for k, r in enumerate(reqs)],
                  views=_pinned(ctx, [grmp.server.ndofs(*r) for r in reqs]),
                  server=grmp.Server("mg", memory_budget=96 << 30, max_active=512))
    ctx.sync()
    return st


# -------------------------------------------------------------------- pass
def _fetch(vec, out):
    """a device vector into page-locked memory that the program keeps"""
    vec.ctx.check(_abi.lib().grmp_vector_download(vec.h, _abi.dptr(out)))
    return out


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "solve":
        sol = grmp.FEVector(st["fes"])
        grmp.solve(sol, st["pde"], solver=case["solver"], precision=case["precision"], rtol=RTOL)
        return sol.entries()
    if kind == "upload":
        grid = grmp.ExtendableGrid.from_arrays(st["coords"], st["cells"])
        fes = grmp.FESpace(_element(case), grid)
        pde = grmp.PoissonProblem(cell_coefficient=grmp.CellCoefficient(st["kap"]))
        pde.add_rhsdata(0, grmp.LinearForm(grmp.Identity, grmp.DataFunction([1.0])))
        pde.add_boundarydata(0, grmp.InterpolateDirichletBoundary, data=grmp.PolynomialData(st["data"]))
        sol = grmp.FEVector(fes)
        grmp.solve(sol, pde, solver="auto", rtol=RTOL)
        return sol.entries()
    if kind == "assemble":
        st["A"].assemble()
        st["A"].spmv(st["x"], st["y"])
        return _fetch(st["y"], st["out"])
    if kind == "stokes":
        sol = grmp.FEVector(st["spaces"])
        grmp.solve(sol, st["pde"], solver="auto", rtol=RTOL)
        return sol.entries()
    if kind == "heat":
        st["tcs"].advance(HEAT_DT)
        return _fetch(st["X"].vec, st["out"])
    if kind == "newton":
        sol = grmp.FEVector(st["fes"])
        grmp.solve(sol, st["pde"], target_residual=RESIDUAL_NEWTON, nonlinear_maxiterations=12, rtol=RTOL_NEWTON)
        return sol.entries()
    srv = st["server"]
    tickets = [srv.submit(k, fe, n, s, rtol=RTOL_SERVED, out=v) for (k, fe, n, s), v in zip(st["reqs"], st["views"])]
    for t in tickets:
        if srv.wait(t).status != 0:
            raise RuntimeError("a served request failed")
    return list(st["views"])


# ----------------------------------------------------------------- accounts
def _sizes(fe, n, ncomp=1):
    """(nodes, cells, dofs, nonzeros) of the generated meshes"""
    if fe == 3:
        m = n + 1
        edges = 3 * m * m * n + 3 * m * n * n + n ** 3
        return m ** 3, 6 * n ** 3, m ** 3, m ** 3 + 2 * edges
    nodes, cells, faces = (n + 1) ** 2, 2 * n * n, 3 * n * n + 2 * n
    if fe == 2:
        # vertex rows meet 7 vertices and 12 faces, face rows 4 vertices and 5 faces (interior)
        return nodes, cells, nodes + faces, nodes * 19 + faces * 9
    return nodes, cells, ncomp * nodes, ncomp * ncomp * nodes * 7


def _mesh_bytes(fe, n):
    nodes, cells, _, _ = _sizes(fe, n)
    dim = 3 if fe == 3 else 2
    return 8 * dim * nodes + 4 * (dim + 1) * cells


def work(case):
    """Inputs read once and outputs written once: mesh, coefficient and data in,
    solution (or product) out; the matrix counts once where the caller keeps it
    (an output of the reassembly, an input of a time step).  Operations: the
    local matrices, and one product with what is assembled."""
    kind, n = case["kind"], case.get("n", 0)
    if kind == "serve":
        b = f = 0.0
        for k, fe, m in _requests(case):
            nodes, cells, dofs, nnz = _sizes(fe, m, 2 if k == 2 else 1)
            b += 8.0 * cells + 8.0 * dofs  # coefficient and solution; the mesh belongs to the shape
            f += cells * 100.0 + 2.0 * nnz
        return {"bytes": b, "flops": f}
    if kind == "stokes":
        nodes, cells = (n + 1) ** 2, 2 * n * n
        dofs = 2 * nodes + 3 * n * n + 2 * n + cells
        return {"bytes": _mesh_bytes(1, n) + 8.0 * dofs, "flops": cells * 2000.0}
    fe = case.get("fe", 1)
    ncomp = 2 if case.get("pde") == "elasticity" else 1
    nodes, cells, dofs, nnz = _sizes(fe, n, ncomp)
    local = {1: 30.0, 2: 250.0, 3: 90.0}[fe] * ncomp * ncomp
    mesh = _mesh_bytes(fe, n) + 8.0 * cells
    if kind == "assemble":
        return {"bytes": mesh + 12.0 * nnz + 16.0 * dofs, "flops": cells * local + 2.0 * nnz}
    if kind == "heat":
        return {"bytes": 12.0 * nnz + 24.0 * dofs, "flops": 4.0 * nnz}
    return {"bytes": mesh + 8.0 * dofs, "flops": cells * local + 2.0 * nnz}


def tolerance(case):
    """Another preconditioner or summation order stops at another error below
    the residual tolerance; a product of reassembled FP64 values differs by
    rounding alone.  About four times the largest difference measured over the
    ranges between a pass and the same problem solved to a much smaller
    residual, or the 64-bit answer: solve 4e-12, upload 4.3e-10 (moved nodes,
    boundary data), Stokes 7e-11, heat 1.3e-11, Newton 2.8e-11, served 4.8e-11,
    product 3e-16."""
    return {"rel": {"solve": 2e-11, "upload": 2e-9, "assemble": 2e-15, "stokes": 3e-10, "heat": 5e-11,
                    "newton": 1e-10, "serve": 2e-10}[case["kind"]]}


# -------------------------------------------------------------- 64-bit answers
_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _t(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), device=_DEV).to(dtype)


def _square(n):
    g = np.arange(n + 1) / n
    X, Y = np.meshgrid(g, g)
    j, i = np.divmod(np.arange(n * n), n)
    v = j * (n + 1) + i
    cells = np.empty((2 * n * n, 3), dtype=np.int64)
    cells[0::2] = np.column_stack([v, v + 1, v + n + 2])
    cells[1::2] = np.column_stack([v, v + n + 2, v + n + 1])
    return np.column_stack([X.ravel(), Y.ravel()]), cells


def _faces(cells, nn):
    """cell faces numbered by first appearance (cell by cell, face (f, f+1)),
    the end nodes of every face, and whether it lies on the boundary"""
    a, b = cells, np.roll(cells, -1, axis=1)
    key = np.minimum(a, b).astype(np.int64) * nn + np.maximum(a, b)
    uniq, first, inv, cnt = np.unique(key.ravel(), return_index=True, return_inverse=True, return_counts=True)
    rank = np.empty(len(uniq), dtype=np.int64)
    order = np.argsort(first)
    rank[order] = np.arange(len(uniq))
    ends = np.column_stack(np.divmod(uniq[order], nn))
    return rank[inv.ravel()].reshape(cells.shape), ends, cnt[order] == 1


def _space(fe, co, cells, ncomp=1):
    """(celldofs, points of the scalar dofs, fixed mask) of P1 / P2 triangles"""
    nn = len(co)
    cf, ends, bnd = _faces(cells, nn)
    fixed = np.zeros(nn, dtype=bool)
    fixed[ends[bnd].ravel()] = True
    dofs, pts = np.asarray(cells, dtype=np.int64), co
    if fe == 2:
        dofs = np.concatenate([dofs, nn + cf], axis=1)
        pts = np.concatenate([co, 0.5 * (co[ends[:, 0]] + co[ends[:, 1]])])
        fixed = np.concatenate([fixed, bnd])
    if ncomp == 2:
        dofs = np.concatenate([dofs, dofs + len(pts)], axis=1)
        fixed = np.concatenate([fixed, fixed])
    return dofs, pts, fixed


def _triangles(co, cells):
    """gradients of the barycentric coordinates (ncells, 3, 2) and areas"""
    X = _t(co)[_t(cells, torch.int64)]
    e1, e2 = X[:, 1] - X[:, 0], X[:, 2] - X[:, 0]
    det = e1[:, 0] * e2[:, 1] - e2[:, 0] * e1[:, 1]
    g1 = torch.stack([e2[:, 1], -e2[:, 0]], 1) / det[:, None]
    g2 = torch.stack([-e1[:, 1], e1[:, 0]], 1) / det[:, None]
    return torch.stack([-g1 - g2, g1, g2], 1), det.abs() / 2


def _tets(co, cells):
    X = _t(co)[_t(cells, torch.int64)]
    e = X[:, 1:] - X[:, :1]
    c = torch.stack([torch.linalg.cross(e[:, 1], e[:, 2]), torch.linalg.cross(e[:, 2], e[:, 0]),
                     torch.linalg.cross(e[:, 0], e[:, 1])], 1)
    det = (e[:, 0] * c[:, 0]).sum(1)
    g = c / det[:, None, None]
    return torch.cat([-g.sum(1, keepdim=True), g], 1), det.abs() / 6


def _gram(G, w):
    """w * G G^T per cell (elementwise products, no batched library call)"""
    return (G[:, :, None, :] * G[:, None, :, :]).sum(-1) * w[:, None, None]


def _p2_gradients(G, q):
    """gradients of the six P2 functions at the midpoint of face q"""
    l = [0.0, 0.0, 0.0]
    l[q], l[(q + 1) % 3] = 0.5, 0.5
    v = [G[:, k] * (4.0 * l[k] - 1.0) for k in range(3)]
    f = [4.0 * (l[k] * G[:, (k + 1) % 3] + l[(k + 1) % 3] * G[:, k]) for k in range(3)]
    return torch.stack(v + f, 1)


def _stiffness(pde, fe, co, cells, kap):
    """(local matrices, local loads of f = 1 per component)"""
    if fe == 3:
        G, vol = _tets(co, cells)
        return _gram(G, kap * vol), (vol / 4)[:, None].expand(-1, 4)
    G, area = _triangles(co, cells)
    if pde == "elasticity":
        mu, lam = 1.0 / 2.6, 0.3 / (1.3 * 0.4)
        z = torch.zeros_like(G[:, :, 0])
        B0 = torch.cat([G[:, :, 0], z], 1)          # eps_xx of the six dofs
        B1 = torch.cat([z, G[:, :, 1]], 1)          # eps_yy
        B2 = torch.cat([G[:, :, 1], G[:, :, 0]], 1)  # 2 eps_xy
        o = lambda a, b: a[:, :, None] * b[:, None, :]  # noqa: E731
        K = (lam + 2 * mu) * (o(B0, B0) + o(B1, B1)) + lam * (o(B0, B1) + o(B1, B0)) + mu * o(B2, B2)
        return K * (kap * area)[:, None, None], (area / 3)[:, None].expand(-1, 3)
    if fe == 1:
        return _gram(G, kap * area), (area / 3)[:, None].expand(-1, 3)
    K = sum(_gram(_p2_gradients(G, q), kap * area / 3) for q in range(3))
    return K, torch.cat([torch.zeros_like(G[:, :, 0]), (area / 3)[:, None].expand(-1, 3)], 1)


def _csr(K, dofs, n):
    nl = dofs.shape[1]
    i = dofs[:, :, None].expand(-1, nl, nl).reshape(-1)
    j = dofs[:, None, :].expand(-1, nl, nl).reshape(-1)
    return torch.sparse_coo_tensor(torch.stack([i, j]), K.reshape(-1), (n, n)).coalesce().to_sparse_csr()


def _cg(A, diag, b, free, x0=None):
    """Jacobi CG on the free dofs to the 64-bit floor, b already lifted"""
    x = torch.zeros_like(b)
    d = torch.where(free, 1.0 / diag, torch.zeros_like(diag))
    for _ in range(3):  # restarts from the true residual
        r = torch.where(free, b - A @ x, torch.zeros_like(b))
        z = d * r
        p = z.clone()
        rz = torch.dot(r, z)
        stop = (r.norm() * 1e-15).item()
        for it in range(100000):
            q = torch.where(free, A @ p, torch.zeros_like(p))
            al = rz / torch.dot(p, q)
            x += al * p
            r -= al * q
            z = d * r
            new = torch.dot(r, z)
            p = z + (new / rz) * p
            rz = new
            if it % 64 == 63 and not r.norm().item() > stop + 1e-14 * b.norm().item():
                break
    return x


def _affordable(fe, n, per):
    """whether some `per` n Jacobi CG iterations in plain torch stay below about 15 seconds"""
    _, _, dofs, nnz = _sizes(fe, n)
    return 3.0 * per * n * (2e-4 + 12.0 * nnz / 3e12 + 100.0 * dofs / 3e12) < 15.0


def _solve_exact(case, co, cells, kap, rhs, bc=None):
    ncomp = 2 if case.get("pde") == "elasticity" else 1
    fe = case["fe"]
    if fe == 3:
        dofs, pts = np.asarray(cells, dtype=np.int64), None
        m = case["n"] + 1
        ijk = np.stack(np.unravel_index(np.arange(m ** 3), (m, m, m)))
        fixed = ((ijk == 0) | (ijk == m - 1)).any(0)
    else:
        dofs, pts, fixed = _space(fe, co, cells, ncomp)
    n = len(fixed)
    D = _t(dofs, torch.int64)
    K, L = _stiffness(case.get("pde", "poisson"), fe, co, cells, kap)
    A = _csr(K, D, n)
    nl = K.shape[1]
    diag = torch.zeros(n, dtype=torch.float64, device=_DEV)
    diag.index_add_(0, D.reshape(-1), torch.diagonal(K, dim1=1, dim2=2).reshape(-1))
    b = torch.zeros_like(diag)
    for c in range(ncomp):
        b.index_add_(0, D[:, c * nl // ncomp:(c + 1) * nl // ncomp].reshape(-1), (rhs[c] * L).reshape(-1))
    free = torch.as_tensor(~fixed, device=_DEV)
    lift = torch.zeros_like(b)
    if bc is not None:
        P = _t(pts)
        g = sum(float(c) * P[:, 0] ** i * P[:, 1] ** j
                for c, (i, j) in zip(bc, ((0, 0), (1, 0), (0, 1), (2, 0), (1, 1), (0, 2))))
        lift = torch.where(free, torch.zeros_like(g), g)
        b = b - A @ lift
    return (lift + _cg(A, diag, b, free)).cpu().numpy()


def exact(case, seed):
    kind, n = case["kind"], case.get("n", 0)
    if kind == "solve":
        if not _affordable(case["fe"], n, {1: 5, 2: 12, 3: 6}[case["fe"]]):
            return None
        grid = _grid(case, seed)
        co, cells = grid.download() if case["fe"] == 3 else _square(n)
        if case["coef"]:
            kap = _t(_kappa(case, seed, len(cells)).download())
        else:
            kap = torch.full((len(cells),), 1e-3 if case["pde"] == "poisson" else 1.0, dtype=torch.float64, device=_DEV)
        rhs = [0.0, -_scale(seed)] if case["pde"] == "elasticity" else [_scale(seed)]
        return _solve_exact(case, co, cells, kap, rhs)
    if kind == "upload":
        co, cells = _triangle_mesh(n, seed)
        kap = _t(np.exp(0.5 * np.random.default_rng(seed + 3).standard_normal(len(cells))))
        return _solve_exact(case, co, cells, kap, [1.0], bc=_quadratic(seed))
    if kind == "assemble":
        grid = _grid(case, seed)
        co, cells = grid.download() if case["fe"] == 3 else _square(n)
        kap = _t(_kappa(case, seed, len(cells)).download())
        ncomp = 2 if case["pde"] == "elasticity" else 1
        dofs = np.asarray(cells, dtype=np.int64) if case["fe"] == 3 else _space(case["fe"], co, cells, ncomp)[0]
        nd = _sizes(case["fe"], n, ncomp)[2]
        xv = grmp.DeviceVector(grmp.default_context(), nd)
        xv.lognormal(seed + 29, 0.0, 1.0)
        x, y = _t(xv.download()), torch.zeros(nd, dtype=torch.float64, device=_DEV)
        for c0 in range(0, len(cells), 4000000):  # in pieces: the local matrices of all cells are large
            s = slice(c0, c0 + 4000000)
            K, _ = _stiffness(case["pde"], case["fe"], co, cells[s], kap[s])
            D = _t(dofs[s], torch.int64)
            y.index_add_(0, D.reshape(-1), (K * x[D][:, None, :]).sum(-1).reshape(-1))
        return y.cpu().numpy()
    if kind == "heat":
        co, cells = _square(n)
        kap = _t(_kappa(case, seed, len(cells)).download())
        dofs, _, fixed = _space(1, co, cells)
        D = _t(dofs, torch.int64)
        G, area = _triangles(co, cells)
        M = area[:, None, None] / 12.0 * (1.0 + torch.eye(3, dtype=torch.float64, device=_DEV))
        K = _gram(G, kap * area) + M / HEAT_DT
        free = torch.as_tensor(~fixed, device=_DEV)
        u = torch.where(free, _t(_initial_heat(n, seed)), torch.zeros(len(fixed), dtype=torch.float64, device=_DEV))
        diag, b = torch.zeros_like(u), torch.zeros_like(u)
        diag.index_add_(0, D.reshape(-1), torch.diagonal(K, dim1=1, dim2=2).reshape(-1))
        b.index_add_(0, D.reshape(-1), ((M * u[D][:, None, :]).sum(-1) / HEAT_DT + area[:, None] / 3.0).reshape(-1))
        return _cg(_csr(K, D, len(fixed)), diag, b, free).cpu().numpy()
    if kind == "newton":
        if case["fe"] == 1:
            return None  # P1 does not hold the bilinear solution: only a nonlinear solve gives its values
        co, cells = _square(n)
        P = _space(2, co, cells)[1]
        a, b, c, d = _bilinear(seed)
        return a + b * P[:, 0] + c * P[:, 1] + d * P[:, 0] * P[:, 1]
    if kind == "serve":
        out = []
        for k, (knd, fe, m) in enumerate(_requests(case)):
            if m > 96:
                out.append(None)  # the small ones stand for the rest: all of them would take minutes
                continue
            co, cells = _square(m)
            kv = grmp.DeviceVector(grmp.default_context(), len(cells))
            kv.lognormal(_request_seed(seed, k), 0.0, 1.0)
            c = dict(fe=fe, n=m, pde="elasticity" if knd == 2 else "poisson")
            out.append(_solve_exact(c, co, cells, _t(kv.download()), [0.0, -1.0] if knd == 2 else [1.0]))
        return out
    return None  # Stokes: a saddle point of this size takes minutes without a multigrid method
