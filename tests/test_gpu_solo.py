"""Even batches of field-grid propagations, which run on one workgroup each,
against the oracle in each class and for a linear medium (whose lengths cannot be
told apart): equal step counts, spectral-energy error of states and saves within
the 1e-6 of the other propagation tests, instances with and without statistics
side by side, and the same bits on a second run.  The first step is 2 mm: at the
default first step the error estimate is rounding noise, and it sets the second
step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def spec_err(a, b):
    pa, pb = np.abs(a) ** 2, np.abs(b) ** 2
    return np.linalg.norm(pa - pb) / np.linalg.norm(pb)


@pytest.mark.parametrize("trange,n,nonlinear", [(0.25e-12, 200, True), (0.5e-12, 256, True), (1e-12, 257, True),
                                                (0.25e-12, 256, False)])
def test_even_batches(trange, n, nonlinear, pkg, capi, orc):
    print(f"case: even batch {trange} {n} {nonlinear}", flush=True)
    from luna_jl_amd import configs, runtime, stats
    kw = {} if nonlinear else dict(kerr=False, plasma=False)
    c = configs.capillary_instance(energy=80e-6, pressure=1.0, trange=trange, flength=0.1, ppt_n=2 ** 12, **kw)
    opts = capi.rk_opts(0.1, save_n=3, init_dz=2e-3)
    ctxs = [runtime.Context(c.holder) for _ in range(n)]
    for ctx in ctxs[3::5]:
        ctx.set_step_stats(stats.StatsFun(c.grid, c.transform, capacity=256))
    E0 = [c.Ew0 * (1.0 + 1e-4 * (i % 7)) for i in range(n)]
    rb = runtime.ResidentBatch(ctxs, E0)
    st = rb.solve(opts)
    first = [rb.state(i) for i in range(n)]
    assert all(s.status == 0 for s in st)
    for i in (0, 3, n - 1):
        code, E, sv, zs, s = orc.solve(c.holder, E0[i], opts)
        assert s.steps == st[i].steps and s.rejected == st[i].rejected
        assert spec_err(first[i], E) <= 1e-6
        assert spec_err(rb.saves(i)[0], sv) <= 1e-6
    assert all(np.array_equal(first[i], first[i % 7]) for i in range(n))
    st2 = rb.solve(opts)
    assert [s.steps for s in st2] == [s.steps for s in st]
    assert all(np.array_equal(rb.state(i), first[i]) for i in range(n))
