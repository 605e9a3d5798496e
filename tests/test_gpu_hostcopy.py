"""Saves of 16 MiB and more leave the device through a ring of page-locked slots
(lh_get_saves, lh_solve); smaller ones and page-locked destinations through one
copy.  Each size around the limit and around a whole number of slots gives the
same bytes on both ways, also into an array that starts inside a page, and
nothing is written around it."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("saves", [31, 32, 33, 64])  # 15.5, 16.03, 16.5 and 32.06 MiB of 513 × 64 bins
def test_large_saves_bytes(saves, pkg):
    print(f"case: {saves} saves", flush=True)
    from luna_jl_amd import _capi, configs, runtime
    inst = configs.radial_instance(N=64, trange=0.25e-12, flength=0.002)
    ctx = runtime.Context(inst.holder)
    opts = _capi.rk_opts(0.002, save_n=saves, init_dz=1e-4)
    _, sv, _, _ = ctx.solve(inst.Ew0, opts)
    n = sv.size
    lib = _capi.lib()
    ptr = C.c_void_p()
    _capi.check(lib.lh_host_alloc(n * 16, C.byref(ptr)), "lh_host_alloc")
    try:
        locked = np.ctypeslib.as_array(C.cast(ptr, C.POINTER(C.c_double)), shape=(2 * n,)).view(np.complex128)
        zs = np.zeros(saves)
        _capi.check(lib.lh_get_saves(ctx.handle, _capi._ptr(locked), _capi._ptr(zs)), "lh_get_saves")
        assert np.array_equal(sv.reshape(-1).view(np.uint64), locked.view(np.uint64))
        assert np.any(sv[-1] != 0)
        pad = np.full(n + 6, 7.0 + 7.0j)
        _capi.check(lib.lh_get_saves(ctx.handle, _capi._ptr(pad[3:-3]), _capi._ptr(zs)), "lh_get_saves")
        assert np.array_equal(pad[3:-3].view(np.uint64), locked.view(np.uint64))
        assert np.all(pad[:3] == 7.0 + 7.0j) and np.all(pad[-3:] == 7.0 + 7.0j)
    finally:
        _capi.check(lib.lh_host_free(ptr), "lh_host_free")
