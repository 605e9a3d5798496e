"""Which kernels a batch runs on: the batches of test_gpu_gang_dense.py,
test_gpu_solo.py and test_gpu_solo_kinds.py reach the kernels they are about."""
import pytest

import test_gpu_gang_dense
import test_gpu_solo_kinds

pytestmark = pytest.mark.gpu


def kinds_of(holders, fields, opts):
    from luna_jl_amd import runtime
    rb = runtime.ResidentBatch([runtime.Context(h) for h in holders], fields)
    assert all(s.status == 0 for s in rb.solve(opts, want_saves=False))
    return runtime.last_launch_kinds()


@pytest.mark.parametrize("n", [177, 300])
def test_uneven(pkg, capi, n):
    print(f"case: kinds of an uneven batch of {n}", flush=True)
    from luna_jl_amd import configs
    insts = test_gpu_gang_dense._batch(configs, n)
    k = kinds_of([c.holder for c in insts], [c.Ew0 for c in insts], capi.rk_opts(2e-4, save_n=2, init_dz=2e-4))
    assert {k[c] for c in (4096, 8192, 16384)} == {capi.LH_KIND_GANG_DENSE}
    assert {v for c, v in k.items() if str(c).startswith("env")} == {capi.LH_KIND_GANG}


@pytest.mark.parametrize("trange,n,nonlinear", [(0.25e-12, 200, True), (0.5e-12, 256, True), (1e-12, 257, True),
                                                (0.25e-12, 256, False)])
def test_even_field(pkg, capi, trange, n, nonlinear):
    print(f"case: kinds of an even batch {trange} {n}", flush=True)
    from luna_jl_amd import configs
    kw = {} if nonlinear else dict(kerr=False, plasma=False)
    c = configs.capillary_instance(energy=80e-6, pressure=1.0, trange=trange, flength=0.1, ppt_n=2 ** 12, **kw)
    E0 = [c.Ew0 * (1.0 + 1e-4 * (i % 7)) for i in range(n)]
    assert list(kinds_of([c.holder] * n, E0, capi.rk_opts(2e-3, save_n=2, init_dz=2e-3)).values()) == [capi.LH_KIND_ALONE]


@pytest.mark.parametrize("make,n", [(lambda: test_gpu_solo_kinds._molecular(0.25e-12), 200),
                                    (lambda: test_gpu_solo_kinds._molecular(0.5e-12), 256),
                                    (test_gpu_solo_kinds._envelope, 257)])
def test_even_kinds(pkg, capi, make, n):
    print(f"case: kinds of an even batch of {n}", flush=True)
    holder, E0, _, dz = make()
    assert list(kinds_of([holder] * n, [E0] * n, capi.rk_opts(dz, save_n=2, init_dz=dz)).values()) == [capi.LH_KIND_ALONE]


def test_others(pkg, capi):
    print("case: kinds of single instances", flush=True)
    from luna_jl_amd import configs
    c = configs.capillary_instance(trange=0.25e-12, flength=0.1, ppt_n=2 ** 12)
    z = test_gpu_solo_kinds._molecular(0.25e-12)
    opts = capi.rk_opts(1e-3, save_n=2, init_dz=1e-3)
    assert kinds_of([c.holder], [c.Ew0], opts) == {4096: capi.LH_KIND_GANG}
    assert kinds_of([c.holder, z[0]], [c.Ew0, z[1]], opts) == {4096: capi.LH_KIND_GANG}
    r = configs.radial_instance(flength=0.1, energy=50e-6, propz=-0.05, R=1.5e-3, N=64, trange=0.3e-12)
    assert kinds_of([r.holder, c.holder], [r.Ew0, c.Ew0], opts) == {"radial": capi.LH_KIND_RADIAL, 4096: capi.LH_KIND_GANG}


@pytest.mark.parametrize("make,most", [(4096, 64), (8192, 64), (16384, 127), ("N2", 64), ("env", 128)])
def test_even_batches_on_each_side(pkg, capi, make, most):
    """Equal instances stay on gangs while those take them in one round (in two
    where a round is short enough), and go to one workgroup each above."""
    print(f"case: kinds at {most} and {most + 1} equal instances, {make}", flush=True)
    from luna_jl_amd import configs
    if make == "N2":
        holder, E0, _, dz = test_gpu_solo_kinds._molecular(0.25e-12)
    elif make == "env":
        holder, E0, _, dz = test_gpu_solo_kinds._envelope()
    else:
        c = configs.capillary_instance(trange={4096: 0.25e-12, 8192: 0.5e-12, 16384: 1e-12}[make], flength=0.1, ppt_n=2 ** 12)
        holder, E0, dz = c.holder, c.Ew0, 2e-3
    for n, kind in [(most, capi.LH_KIND_GANG), (most + 1, capi.LH_KIND_ALONE)]:
        assert list(kinds_of([holder] * n, [E0] * n, capi.rk_opts(dz, save_n=2, init_dz=dz)).values()) == [kind], n


@pytest.mark.parametrize("init_dz", [1e-4, 2e-3])
def test_even_batch_against_one(pkg, capi, init_dz):
    """An instance of an even batch (one workgroup) and the same one solved by
    itself (a gang) take the same steps and agree to the propagation tests' 1e-6
    in spectral energy, also with the default first step, whose error estimate is
    rounding noise and sets the next step."""
    print(f"case: even batch against one, first step {init_dz}", flush=True)
    import numpy as np
    from luna_jl_amd import configs, runtime
    c = configs.capillary_instance(energy=80e-6, pressure=1.0, trange=0.5e-12, flength=0.1, ppt_n=2 ** 12)
    opts = capi.rk_opts(0.1, save_n=5, init_dz=init_dz)
    ctxs = [runtime.Context(c.holder) for _ in range(65)]
    states, saves, _, st = runtime.batch_solve(ctxs, [c.Ew0] * 65, opts)
    assert runtime.last_launch_kinds() == {8192: capi.LH_KIND_ALONE}
    E, sv, _, s = ctxs[0].solve(c.Ew0, opts)
    assert runtime.last_launch_kinds() == {8192: capi.LH_KIND_GANG}

    def err(a, b):
        a, b = np.abs(a) ** 2, np.abs(b) ** 2
        return np.linalg.norm(a - b) / np.linalg.norm(b)

    assert (st[64].steps, st[64].rejected) == (s.steps, s.rejected)
    assert err(states[64], E) <= 1e-6 and err(saves[64], sv) <= 1e-6


def test_kinds_of_grid_beside_each_other(pkg, capi):
    """Field and envelope instances in one batch, whose estimated costs cannot be
    compared: both on gangs, and together about as long as one after the other."""
    print("case: 40 envelope instances beside 100 field ones", flush=True)
    from luna_jl_amd import configs, runtime
    c = configs.capillary_instance(energy=80e-6, pressure=1.0, trange=1e-12, flength=0.1, ppt_n=2 ** 12)
    g = configs.gnlse_instance(trange=6e-12, flength=0.005)
    parts = [(c.holder, c.Ew0, capi.rk_opts(0.05, save_n=2, init_dz=2e-3))] * 100
    parts += [(g.holder, g.Ew0, capi.rk_opts(0.001, save_n=2, init_dz=1e-4))] * 40
    ctxs = [runtime.Context(h) for h, _, _ in parts]

    def ms(sel):
        run = lambda: runtime.batch_solve_opts([ctxs[i] for i in sel], [parts[i][1] for i in sel], [parts[i][2] for i in sel], want_saves=False)
        run()
        assert all(s.status == 0 for s in run()[3])
        return max(t for t, _ in runtime.last_launch_times().values())

    field, env, both = ms(range(100)), ms(range(100, 140)), ms(range(140))
    print(f"ms: {field:.2f} {env:.2f} {both:.2f}", flush=True)
    assert runtime.last_launch_kinds() == {16384: capi.LH_KIND_GANG, "env8192": capi.LH_KIND_GANG}
    assert both <= 2 * (field + env)


def test_kinds_that_cannot_be_compared(pkg, capi):
    """Even instances go to one workgroup each only where all of the batch are of
    one kind: with a Raman gas or an envelope grid beside them they stay on gangs."""
    print("case: even instances beside others", flush=True)
    from luna_jl_amd import configs
    c = configs.capillary_instance(energy=80e-6, pressure=1.0, trange=0.25e-12, flength=0.1, ppt_n=2 ** 12)
    opts = capi.rk_opts(1e-3, save_n=2, init_dz=1e-3)
    assert kinds_of([c.holder] * 100, [c.Ew0] * 100, opts) == {4096: capi.LH_KIND_ALONE}
    raman, env = test_gpu_solo_kinds._molecular(0.25e-12), test_gpu_solo_kinds._envelope()
    assert kinds_of([c.holder] * 100 + [raman[0]], [c.Ew0] * 100 + [raman[1]], opts) == {4096: capi.LH_KIND_GANG}
    k = kinds_of([c.holder] * 100 + [env[0]], [c.Ew0] * 100 + [env[1]], opts)
    assert k == {4096: capi.LH_KIND_GANG, "env4096": capi.LH_KIND_GANG}
