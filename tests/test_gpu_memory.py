"""Device memory: what objects give back, and what the pool of freed blocks
holds (grmp_pool_usage is for these tests; it is not in include/grmp.h)."""
import ctypes
import gc

import pytest

pytestmark = pytest.mark.gpu


def _usage(grmp, ctx):
    ctx.sync()
    used, held = ctypes.c_int64(), ctypes.c_int64()
    f = grmp.lib().grmp_pool_usage
    f.argtypes, f.restype = [ctypes.c_void_p] + [ctypes.POINTER(ctypes.c_int64)] * 2, ctypes.c_int
    ctx.check(f(ctx.h, ctypes.byref(used), ctypes.byref(held)))
    return used.value, held.value


def test_destroyed_matrices_give_everything_back(grmp):
    """After the first one (which grows the context's scratch and leaves its
    table of forms for the next) a matrix's life leaves no byte of the pool in
    use."""
    print("[case] matrices created, assembled and destroyed", flush=True)
    gc.collect()  # what other tests left behind
    grid = grmp.grid_unitsquare(9)
    fes = grmp.FESpace(grmp.H1P1(1), grid)
    used = []
    for _ in range(4):
        A = grmp.FEMatrix([fes])
        form, keep = grmp.LaplaceOperator(1.0).form(fes, 0, 0, fes.ctx)
        A.add_form(form, keep)
        A.build_pattern()
        A.assemble()
        del A, form, keep
        used.append(_usage(grmp, fes.ctx)[0])
    assert used[1:] == used[1:2] * 3, used


def test_contexts_share_their_freed_blocks(grmp):
    """256 MiB freed by one context serve another, and go back when one of them
    is destroyed.  (A pool for each context held 512 MiB here.)"""
    print("[case] two contexts", flush=True)
    size = 256 << 20
    gc.collect()
    A, B = grmp._abi.Context(0), grmp._abi.Context(0)
    used0, held0 = _usage(grmp, A)
    for ctx in (A, B):
        v = grmp.DeviceVector(ctx, size // 8)
        u, h = _usage(grmp, ctx)
        assert u >= used0 + size and h < held0 + size + size // 2, (used0, held0, u, h)
        del v
        gc.collect()
        assert _usage(grmp, ctx)[0] == used0
    assert _usage(grmp, A)[1] >= size  # kept for the next call
    B.close()
    assert _usage(grmp, A)[1] < held0 + size // 2
    A.close()


def test_closed_server_gives_its_memory_back(grmp):
    """Nothing in use and no freed block held after a server of ten contexts"""
    print("[case] memory after a server", flush=True)
    ctx = grmp._abi.default_context()
    gc.collect()
    grmp._abi.Context(0).close()  # what earlier tests left free
    used0, held0 = _usage(grmp, ctx)
    with grmp.Server("mg", memory_budget=64 << 20) as S:
        ts = [S.submit(1 + k % 2, 1, 100 + k, k) for k in range(24)]
        assert all(S.wait(t).status == 0 for t in ts)
        assert _usage(grmp, ctx)[1] > held0
    used1, held1 = _usage(grmp, ctx)
    assert used1 == used0 and held1 <= held0, (used0, held0, used1, held1)


def _levels(grmp, kind, fe, N):
    """(matrix, space, mesh) of a multigrid request's levels"""
    shape = [(fe, N)] + ([(1, N)] if fe == 2 else [])
    while N > 4:
        N = (N + 1) // 2
        shape.append((1, N))
    out = []
    for f, n in shape:
        grid = grmp.grid_unitsquare(n)
        fes = grmp.FESpace(grmp.H1P2(1) if f == 2 else grmp.H1P1(kind), grid)
        op = grmp.LaplaceOperator(1.0) if kind == 1 else grmp.HookStiffnessOperator2D(1.0, 1.0)
        A = grmp.FEMatrix([fes])
        A.add_form(*op.form(fes, 0, 0, fes.ctx))
        A.set_fixed(fes.boundary_dofs(), 1e60)
        A.build_pattern()
        out.append((A, fes, grid))
    return out


# one workgroup's LDS image with and without all levels (1,250 rows of
# elasticity do not fit), the largest that run whole in one workgroup (P1 44, P2
# 22, elasticity 31), one level
@pytest.mark.parametrize("kind,fe,N", [(1, 1, 2), (1, 1, 4), (1, 1, 16), (1, 1, 35), (1, 1, 44), (1, 1, 64), (1, 1, 200),
                                       (1, 2, 1), (1, 2, 9), (1, 2, 22), (1, 2, 40), (2, 1, 3), (2, 1, 16), (2, 1, 24),
                                       (2, 1, 31), (2, 1, 64)])
def test_multigrid_buffer_is_within_its_account(grmp, kind, fe, N):
    """What a hierarchy allocates is at most what the server reserves for such a
    request, and at most mg_job_bytes of its actual nonzeros.  (With the LDS
    image at its largest size for all, P1 16x16 took 240 KB of 92 reserved.)"""
    print(f"[case] multigrid buffer {kind} {fe} {N}", flush=True)
    gc.collect()
    lv = _levels(grmp, kind, fe, N)
    ctx = lv[0][1].ctx
    kappa0 = grmp.DeviceVector(ctx, lv[0][2].ncells)
    kappa0.fill(1.0)
    used0 = _usage(grmp, ctx)[0]
    M = grmp.MultigridSolver(lv, kappa0)
    taken = _usage(grmp, ctx)[0] - used0
    del M

    L = grmp.lib()
    L.mg_request_reserve.restype = L.mg_job_bytes.restype = ctypes.c_int64
    req = grmp.server.request(kind, fe, N, 1)
    reserve = L.mg_request_reserve(ctypes.byref(req), 2048, 2048)
    k = len(lv)
    arr = lambda t, v: (t * k)(*v)
    info = [a.info() for a, _, _ in lv]
    bound = L.mg_job_bytes(k, arr(ctypes.c_int64, [i[0] for i in info]), arr(ctypes.c_int64, [i[1] for i in info]),
                           arr(ctypes.c_int64, [g.ncells for _, _, g in lv]), arr(ctypes.c_int, [g.N for _, _, g in lv]),
                           2048, 2048)
    assert 0 < taken <= bound <= reserve, (taken, bound, reserve)
    assert reserve >= 2 * grmp.server.footprint(kind, fe, N)


def test_out_of_memory_gives_free_blocks_back(grmp):
    """A vector larger than the device fails with the library's code after the
    free blocks were given back for it, and the context works on."""
    print("[case] a vector larger than the device", flush=True)
    size = 256 << 20
    gc.collect()
    ctx = grmp._abi.Context(0)
    v = grmp.DeviceVector(ctx, size // 8)
    del v
    gc.collect()
    assert _usage(grmp, ctx)[1] >= size
    with pytest.raises(grmp.GrmpError) as e:
        grmp.DeviceVector(ctx, 1 << 40)
    assert e.value.code == grmp._abi.ERR_OOM
    used, held = _usage(grmp, ctx)
    assert held - used < size
    w = grmp.DeviceVector(ctx, 1000)
    w.fill(2.0)
    assert (w.download() == 2.0).all()
    del w
    ctx.close()
