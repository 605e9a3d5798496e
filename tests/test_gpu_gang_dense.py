"""Batches large enough for the kernels that run two workgroups on a CU: every
instance equals the same instance solved alone, bit for bit, in each class that
has such a kernel, with a class that has none beside them and with the per-step
statistics on."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(configs, n):
    rng = np.random.default_rng(5)
    out = []
    for i in range(n):
        if i % 12 == 11:
            out.append(configs.gnlse_instance(trange=(3e-12, 6e-12, 12e-12)[i // 12 % 3], flength=0.01, noise_seed=i))
        else:
            out.append(configs.capillary_instance(energy=float(rng.uniform(40e-6, 120e-6)), pressure=1.0 + 0.002 * i,
                                                  trange=(0.25e-12, 0.5e-12, 1e-12)[i % 3], flength=0.01,
                                                  ppt_n=2 ** 12))
    return out


@pytest.mark.parametrize("n", [177, 300])  # the first of them; more instances than their gangs
def test_large_batches(pkg, capi, n):
    print(f"case: batch of {n}", flush=True)
    from luna_jl_amd import configs, runtime, stats
    insts = _batch(configs, n)
    opts = capi.rk_opts(0.002, save_n=3, init_dz=2e-4)

    def context(c, i):
        ctx = runtime.Context(c.holder)
        if i % 12 == 3:
            ctx.set_step_stats(stats.StatsFun(c.grid, c.transform, capacity=64))
        return ctx

    ctxs = [context(c, i) for i, c in enumerate(insts)]
    states, saves, _, st = runtime.batch_solve(ctxs, [c.Ew0 for c in insts], opts)
    assert all(s.status == 0 for s in st)
    classes = set()
    for i in list(range(0, 36)) + [n // 2, n - 1]:
        E, sv, _, s = context(insts[i], i).solve(insts[i].Ew0, opts)
        classes.add((insts[i].grid.n_to, np.iscomplexobj(insts[i].grid.t)))
        assert s.steps == st[i].steps
        assert np.array_equal(E, states[i]) and np.array_equal(sv, saves[i])
    assert len(classes) >= 3
