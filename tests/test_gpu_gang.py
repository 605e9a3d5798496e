"""Batches on gangs of workgroups: every instance of a batch equals the same
instance solved alone, bit for bit, for batch sizes around the launch's units
(fewer instances than gangs, one more than a multiple of eight, more instances
than gangs) and with kernels of several kinds side by side; one right-hand
side per size class against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _instances(configs, n, flength=0.01):
    rng = np.random.default_rng(5)
    out = []
    for i in range(n):
        out.append(configs.capillary_instance(energy=float(rng.uniform(40e-6, 120e-6)), pressure=1.0 + 0.01 * i,
                                              trange=0.25e-12 if i % 3 else 0.5e-12, flength=flength, ppt_n=2 ** 12))
    return out


@pytest.mark.parametrize("n", [2, 9, 70])
def test_batch_sizes(pkg, capi, n):
    from luna_jl_amd import configs, runtime
    insts = _instances(configs, n)
    opts = capi.rk_opts(0.01, save_n=3)
    states, saves, _, stats = runtime.batch_solve([runtime.Context(c.holder) for c in insts],
                                                  [c.Ew0 for c in insts], opts)
    assert all(s.status == 0 for s in stats)
    for i in {0, 1, n // 2, n - 1}:
        E, sv, _, st = runtime.Context(insts[i].holder).solve(insts[i].Ew0, opts)
        assert st.steps == stats[i].steps
        assert np.array_equal(E, states[i]) and np.array_equal(sv, saves[i])


def test_mixed_kernels(pkg, capi):
    """Constant fill, gradient fill and a Raman gas in one batch."""
    from luna_jl_amd import configs, runtime
    from luna_jl_amd.interface import prop_capillary_args

    def cap(gas, pressure, trange):
        Ew, grid, linop, tr, _, _ = prop_capillary_args(
            125e-6, 0.01, gas, pressure, lambda0=800e-9, lambda_lims=(150e-9, 4e-6), trange=trange,
            tau_fwhm=10e-15, energy=40e-6, shotnoise=False, ppt_N=2 ** 12)
        return tr.descriptor(linop), Ew

    ones = [cap("He", 1.0, 0.5e-12), cap("He", (0.5, 1.0), 0.5e-12), cap("N2", 0.3, 0.25e-12),
            cap("He", 1.0, 0.25e-12)]
    g = configs.gnlse_instance(trange=3e-12, flength=0.01)
    ones.append((g.holder, g.Ew0))
    opts = capi.rk_opts(0.002, save_n=2, init_dz=2e-4)
    ctxs = [runtime.Context(h) for h, _ in ones]
    states, _, _, stats = runtime.batch_solve(ctxs, [E for _, E in ones], opts)
    for (h, E0), got, st in zip(ones, states, stats):
        E, _, _, s = runtime.Context(h).solve(E0, opts)
        assert st.status == 0 and s.steps == st.steps and np.array_equal(E, got)


@pytest.mark.parametrize("trange,kerr,plasma", [(0.25e-12, True, True), (0.5e-12, False, True), (1e-12, True, False)])
def test_rhs_many_ionising_samples(pkg, orc, trange, kerr, plasma):
    """A field that ionises far more samples than the members' lists hold (a
    flat-topped pulse over the whole window): the rates of a lane's own samples."""
    from luna_jl_amd import configs, runtime
    c = configs.capillary_instance(energy=100e-6, pressure=1.0, trange=trange, flength=0.1, ppt_n=2 ** 12, kerr=kerr,
                                   plasma=plasma)
    g = c.grid
    t = np.arange(g.n_t) * (g.t[1] - g.t[0])
    Et = np.cos(2 * np.pi * 3e8 / 800e-9 * t)
    Ew = np.fft.rfft(Et)[:g.n_omega]
    peak = 0.5 * (c.holder.desc.field_div) * 5e10
    Ew = Ew * peak
    nl = runtime.Context(c.holder).rhs(Ew)
    st, ref = orc.rhs(c.holder, Ew)
    assert st == 0
    assert np.linalg.norm(nl - ref) <= 1e-12 * np.linalg.norm(ref)
