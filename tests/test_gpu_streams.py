"""Calls on the caller's streams: a solve without allocations behind other work,
right-hand sides that overlap a solve of the same context."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Hip:
    """Streams and device memory from the HIP runtime that the library links."""

    def __init__(self):
        self.L = C.CDLL("libamdhip64.so.7")
        self.L.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.L.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
        for f in ("hipFree", "hipStreamSynchronize", "hipStreamDestroy"):
            getattr(self.L, f).argtypes = [C.c_void_p]
        self.mem, self.streams = [], []

    def check(self, rc):
        assert rc == 0, rc

    def put(self, a):
        p = C.c_void_p()
        self.check(self.L.hipMalloc(C.byref(p), a.nbytes))
        self.check(self.L.hipMemcpy(p, a.ctypes.data, a.nbytes, 1))
        self.mem.append(p)
        return p

    def get(self, p, like):
        out = np.empty_like(like)
        self.check(self.L.hipMemcpy(out.ctypes.data, p, out.nbytes, 2))
        return out

    def stream(self):
        s = C.c_void_p()
        self.check(self.L.hipStreamCreate(C.byref(s)))
        self.streams.append(s)
        return s

    def sync(self, s):
        self.check(self.L.hipStreamSynchronize(s))

    def close(self):
        for s in self.streams:
            self.L.hipStreamSynchronize(s)
            self.L.hipStreamDestroy(s)
        for p in self.mem:
            self.L.hipFree(p)


@pytest.fixture
def hip(pkg, capi):
    capi.lib()
    h = Hip()
    yield h
    h.close()


def field(n_to, gas="He", pressure=1.0, energy=60e-6):
    from luna_jl_amd.interface import prop_capillary_args
    Ew, grid, linop, tr, _, _ = prop_capillary_args(
        125e-6, 0.05, gas, pressure, lambda0=800e-9, lambda_lims=(150e-9, 4e-6),
        trange={4096: 0.25e-12, 8192: 0.5e-12, 16384: 1e-12}[n_to], tau_fwhm=10e-15, energy=energy, shotnoise=False,
        ppt_N=2 ** 12)
    assert grid.n_to == n_to
    return tr.descriptor(linop), np.ascontiguousarray(Ew, dtype=np.complex128)


def rhs(capi, ctx, out, inp, stream, z=0.0):
    capi.check(capi.lib().lh_rhs_device(ctx.handle, out, inp, z, stream), "lh_rhs_device")


def test_noalloc_behind_other_work(hip, capi):
    print("case: lh_solve_noalloc on a stream with work in front", flush=True)
    from luna_jl_amd import runtime
    holder, E0 = field(8192)
    ctx, other = runtime.Context(holder), runtime.Context(holder)
    opts = capi.rk_opts(0.02, save_n=300, init_dz=1e-3)
    E, sv, zs, st = ctx.solve(E0, opts)
    inp, out = hip.put(E0), hip.put(E0)
    state, saves, s = hip.put(E0), hip.put(np.zeros_like(sv)), hip.stream()
    for _ in range(200):
        rhs(capi, other, out, inp, s)
    st2 = capi.LhStats()
    rc = capi.lib().lh_solve_noalloc(ctx.handle, state, C.byref(opts), saves, None, C.byref(st2), s)
    assert rc == 0 and (st2.steps, st2.rejected, st2.saved) == (st.steps, st.rejected, st.saved)
    assert np.array_equal(hip.get(state, E), E) and np.array_equal(hip.get(saves, sv), sv)


@pytest.mark.parametrize("gas,pressure,n_to", [("N2", 0.5, 8192), ("He", (0.5, 1.0), 8192), ("He", 1.0, 4096)])
def test_rhs_beside_a_solve(hip, capi, gas, pressure, n_to):
    """Asynchronous right-hand sides (Raman gas, gradient fill at another z,
    constant fill) and a solve of the same context at the same time."""
    print(f"case: rhs beside a solve, {gas} {pressure}", flush=True)
    from luna_jl_amd import runtime
    holder, E0 = field(n_to, gas, pressure)
    ctx = runtime.Context(holder)
    opts = capi.rk_opts(0.01, save_n=3, init_dz=1e-3)
    E, sv, _, st = ctx.solve(E0, opts)
    nl = ctx.rhs(E0, 0.04)
    inp, out, s = hip.put(E0), hip.put(np.zeros_like(E0)), hip.stream()
    for _ in range(3):
        for _ in range(300):
            rhs(capi, ctx, out, inp, s, 0.04)
        E2, sv2, _, st2 = ctx.solve(E0, opts)
        assert st2.steps == st.steps and np.array_equal(E2, E) and np.array_equal(sv2, sv)
        hip.sync(s)
        assert capi.lib().lh_ctx_status(ctx.handle) == 0
        assert np.array_equal(hip.get(out, nl), nl)
