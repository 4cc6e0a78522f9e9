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
