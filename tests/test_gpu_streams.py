"""Calls on the caller's streams: a solve without allocations behind other work,
right-hand sides that overlap a solve of the same context or each other, and
captured ones."""
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

    def graph(self, s, record):
        """The executable graph of what record() enqueues on s."""
        g, e = C.c_void_p(), C.c_void_p()
        self.check(self.L.hipStreamBeginCapture(s, 2))  # hipStreamCaptureModeRelaxed
        record()
        self.check(self.L.hipStreamEndCapture(s, C.byref(g)))
        self.check(self.L.hipGraphInstantiate(C.byref(e), g, None, None, C.c_size_t(0)))
        self.check(self.L.hipGraphDestroy(g))
        return e

    def event(self):
        e = C.c_void_p()
        self.check(self.L.hipEventCreateWithFlags(C.byref(e), 2))  # hipEventDisableTiming
        return e

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


KINDS = [("N2", 0.5, 8192), ("He", (0.5, 1.0), 8192), ("He", 1.0, 16384)]


@pytest.mark.parametrize("gas,pressure,n_to", KINDS)
def test_rhs_on_many_streams(hip, capi, gas, pressure, n_to):
    """One context on seven streams in turn without a wait between the calls
    (more than it keeps memory for at once), some of them destroyed in between."""
    print(f"case: rhs on many streams, {gas} {pressure}", flush=True)
    from luna_jl_amd import runtime
    holder, E0 = field(n_to, gas, pressure)
    ctx = runtime.Context(holder)
    fields = [E0 * (1 - 0.05 * i) for i in range(7)]
    ref = [ctx.rhs(f, 0.01 * i) for i, f in enumerate(fields)]
    inp, out = [hip.put(f) for f in fields], [hip.put(np.zeros_like(E0)) for _ in fields]
    for _ in range(2):
        streams = [hip.stream() for _ in fields]
        for _ in range(40):
            for i, s in enumerate(streams[:3]):
                rhs(capi, ctx, out[i], inp[i], s, 0.01 * i)
        assert np.array_equal(ctx.rhs(fields[4], 0.04), ref[4])  # its own stream, beside them
        for i, s in enumerate(streams):
            rhs(capi, ctx, out[i], inp[i], s, 0.01 * i)
        for s in streams:
            hip.sync(s)
        assert capi.lib().lh_ctx_status(ctx.handle) == 0
        for i, o in enumerate(out):
            assert np.array_equal(hip.get(o, E0), ref[i]), i
        for s in streams[::2]:
            hip.streams.remove(s)
            hip.check(hip.L.hipStreamDestroy(s))


@pytest.mark.parametrize("gas,pressure,n_to", KINDS)
def test_captured_rhs(hip, capi, gas, pressure, n_to):
    """Captured right-hand sides, on one stream and on a fork of it, replayed
    beside eager ones on another stream and a solve; every replay against the
    eager result."""
    print(f"case: captured rhs, {gas} {pressure}", flush=True)
    from luna_jl_amd import runtime
    holder, E0 = field(n_to, gas, pressure)
    ctx = runtime.Context(holder)
    opts = capi.rk_opts(0.005, save_n=0, init_dz=1e-3)
    E = ctx.solve(E0, opts, want_saves=False)[0]
    fields = [E0, 0.9 * E0, 0.8 * E0]
    ref = [ctx.rhs(f, 0.02) for f in fields]
    inp, out = [hip.put(f) for f in fields], [hip.put(np.zeros_like(E0)) for _ in fields]
    zero = np.zeros_like(E0)
    s, fork, eager = hip.stream(), hip.stream(), hip.stream()
    e1, e2 = hip.event(), hip.event()

    def record():
        rhs(capi, ctx, out[0], inp[0], s, 0.02)
        hip.check(hip.L.hipEventRecord(e1, s))
        hip.check(hip.L.hipStreamWaitEvent(fork, e1, 0))
        rhs(capi, ctx, out[1], inp[1], fork, 0.02)
        rhs(capi, ctx, out[0], inp[0], s, 0.02)
        hip.check(hip.L.hipEventRecord(e2, fork))
        hip.check(hip.L.hipStreamWaitEvent(s, e2, 0))

    hip.L.hipGraphLaunch.argtypes = [C.c_void_p, C.c_void_p]
    for f in ("hipEventRecord", "hipStreamWaitEvent"):
        getattr(hip.L, f).argtypes = [C.c_void_p, C.c_void_p] + ([C.c_uint] if f == "hipStreamWaitEvent" else [])
    g = hip.graph(s, record)
    for k in range(4):
        for o in out:
            hip.check(hip.L.hipMemcpy(o, zero.ctypes.data, zero.nbytes, 1))
        for _ in range(5):
            hip.check(hip.L.hipGraphLaunch(g, s))
            rhs(capi, ctx, out[2], inp[2], eager, 0.02)
        if k % 2:
            assert np.array_equal(ctx.solve(E0, opts, want_saves=False)[0], E)
        hip.sync(s)
        hip.sync(eager)
        for o, r in zip(out, ref):
            assert np.array_equal(hip.get(o, E0), r)
    hip.L.hipGraphExecDestroy(g)
