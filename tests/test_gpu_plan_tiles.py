"""A plan that is set, imported or measured runs with its own number of MFMA tiles,
whatever the size of the grid; the default plan runs with one tile where the
grid has few workgroups.  The tiles move no bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_plans_run_as_set(pkg):
    from luna_jl_amd import configs, runtime
    print("case: tiles of the plans at Nto = 2048, Nr = 64", flush=True)
    runtime.wisdom_forget()
    inst = configs.radial_instance(flength=0.1, energy=50e-6, propz=-0.05, R=1.5e-3, N=64, trange=0.3e-12)
    ctx = runtime.Context(inst.holder)
    assert ctx.plan == (0, 2) and ctx.plan_tiles == 1
    ref = {0: ctx.rhs(inst.Ew0)}
    for fft in (0, 1):
        for mt in (2, 4, 1):
            ctx.plan = (fft, mt)
            assert ctx.plan == (fft, mt) and ctx.plan_tiles == mt
            nl = ctx.rhs(inst.Ew0)
            assert np.array_equal(nl, ref.setdefault(fft, nl))
    try:
        runtime.wisdom_import("luna-hip-wisdom 1\nradial 2048 64 0 2 10.0\n")
        ctx = runtime.Context(inst.holder)
        assert ctx.plan == (0, 2) and ctx.plan_tiles == 2
        runtime.wisdom_forget()
        ctx.autotune(inst.Ew0, reps=2)
        assert ctx.plan_tiles == ctx.plan[1]
    finally:
        runtime.wisdom_forget()


def test_default_tiles_by_size(pkg):
    from luna_jl_amd import configs, runtime
    print("case: default tiles by size", flush=True)
    runtime.wisdom_forget()
    for nr, trange, tiles in [(64, 0.25e-12, 1), (256, 0.25e-12, 1), (64, 1e-12, 1), (192, 0.5e-12, 2), (128, 1e-12, 2)]:
        inst = configs.radial_instance(N=nr, trange=trange)
        ctx = runtime.Context(inst.holder)
        assert ctx.plan == (0, 2) and ctx.plan_tiles == tiles, (nr, inst.grid.n_to)
