"""Device memory: what objects give back, and what the pool of freed blocks
holds (grmp_pool_usage is for these tests; it is not in include/grmp.h)."""
import ctypes

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
    """After the first one (which grows the context's scratch) a matrix's life
    leaves no byte of the pool in use."""
    print("[case] matrices created, assembled and destroyed", flush=True)
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
