"""Even batches that run on one workgroup per instance with a field-grid Raman
response and on the 4096-point envelope grid, against the oracle: equal step
counts, spectral-energy error of states and saves within the 1e-6 of the other
propagation tests, and the same bits for equal instances."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def spec_err(a, b):
    pa, pb = np.abs(a) ** 2, np.abs(b) ** 2
    return np.linalg.norm(pa - pb) / np.linalg.norm(pb)


def _molecular(trange):
    from luna_jl_amd.interface import prop_capillary_args
    Ew, grid, linop, tr, _, _ = prop_capillary_args(125e-6, 0.02, "N2", 0.5, lambda0=800e-9, lambda_lims=(150e-9, 4e-6),
                                                    trange=trange, tau_fwhm=10e-15, energy=40e-6, shotnoise=False,
                                                    ppt_N=2 ** 12)
    return tr.descriptor(linop), Ew, 0.02, 1e-3


def _envelope():
    from luna_jl_amd import configs
    g = configs.gnlse_instance(trange=3e-12, flength=0.005)
    return g.holder, g.Ew0, 0.005, 1e-4


@pytest.mark.parametrize("make,n", [(lambda: _molecular(0.25e-12), 200), (lambda: _molecular(0.5e-12), 256),
                                    (_envelope, 257)])
def test_even_batches(make, n, pkg, capi, orc):
    from luna_jl_amd import runtime
    holder, E0, L, dz = make()
    print(f"case: even batch of {n}", flush=True)
    opts = capi.rk_opts(L, save_n=3, init_dz=dz)
    rb = runtime.ResidentBatch([runtime.Context(holder) for _ in range(n)], [E0] * n)
    st = rb.solve(opts)
    assert all(s.status == 0 for s in st)
    code, E, sv, zs, s = orc.solve(holder, E0, opts)
    for i in (0, n - 1):
        assert s.steps == st[i].steps and s.rejected == st[i].rejected
        assert spec_err(rb.state(i), E) <= 1e-6
        assert spec_err(rb.saves(i)[0], sv) <= 1e-6
    assert all(np.array_equal(rb.state(i), rb.state(0)) for i in range(1, n))
