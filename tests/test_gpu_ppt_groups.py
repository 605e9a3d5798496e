"""lh_ppt_table at the sizes where its launch changes: one value, fewer values
than workgroups, a remainder, the last table with a wavefront per value and the
first with 16 lanes per value, more than 256 values per workgroup; ascending and
descending fields.  Against the host restatement of ionrate_fun_PPT
(src/Ionisation.jl:317-390) at every 251st value and both ends, to the 1e-11
of the full-table test."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 257, 16384, 16385, 65537])
@pytest.mark.parametrize("gas,lam0", [("He", 800e-9), ("Ar", 800e-9)])
def test_table_sizes_match_host(gas, lam0, n, pkg):
    print(f"case: ppt table {gas} n={n}", flush=True)
    from luna_jl_amd import ionisation
    o = ionisation.ppt_options(gas)
    Emax = 2 * ionisation.barrier_suppression(o["ionpot"], o["Z"])
    E = np.linspace(Emax, Emax / 50, n)
    if n % 2:
        E = E[::-1].copy()
    r = ionisation.ppt_device_table(o["ionpot"], lam0, o["Z"], o["l"], E, dalpha=o["dalpha"], alpha_ion=o["alpha_ion"])
    at = np.unique(np.r_[np.arange(0, n, 251), n - 1])
    ref = ionisation.ionrate_ppt_vec(o["ionpot"], lam0, o["Z"], o["l"], E[at], dalpha=o["dalpha"],
                                     alpha_ion=o["alpha_ion"])
    assert np.all(np.isfinite(r))
    m = ref > 1e-300
    assert m.any()
    assert np.max(np.abs(r[at][m] - ref[m]) / ref[m]) <= 1e-11
