"""The surrogate's products at extents that are no whole tiles or vectors: odd
channel tiles (96), one and three input channels, mode counts that leave a row of
the DFT matrices unaligned, a batch of one, a hidden layer of half a tile, a
series shorter than a slab; the gradient against the BF16-operand oracle with the
tolerances of the parity test of the same depth or deeper (four times the effect
of FP32 accumulation order on BF16 rounding)."""
import numpy as np
import pytest

from oracle import fno_oracle

pytestmark = pytest.mark.gpu

SHAPES = [  # dims, batch
    (dict(n_x=64, cin=1, channels=32, modes=5, layers=1, hidden=32), 1),
    (dict(n_x=192, cin=3, channels=96, modes=7, layers=2, hidden=96), 3),
    (dict(n_x=128, cin=2, channels=64, modes=64, layers=2, hidden=160), 5),
    (dict(n_x=1088, cin=4, channels=32, modes=33, layers=2, hidden=64), 4),
]


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, float) - np.asarray(b, float)) / np.linalg.norm(np.asarray(b, float)))


@pytest.mark.parametrize("dims,B", SHAPES)
def test_fno_odd_shapes(dims, B, pkg):
    print(f"case: fno {dims} batch {B}", flush=True)
    from luna_jl_amd import surrogate
    tol_f, tol_g = 1.2e-2, 2e-2
    net = surrogate.FNO(max_batch=B, **dims)
    p = net.init_params(seed=0)
    for name, (o, shape) in net.layout.items():  # make the spectral path carry weight
        if name.startswith("R"):
            p[o:o + int(np.prod(shape))] *= 50.0
    net.set_params(p)
    orc = fno_oracle.FNOOracle(dims["n_x"], dims["cin"], dims["channels"], dims["modes"], dims["layers"], dims["hidden"])
    rng = np.random.default_rng(7)
    x = rng.standard_normal((B, dims["n_x"], dims["cin"])).astype(np.float32)
    t = (0.5 * rng.standard_normal((B, dims["n_x"]))).astype(np.float32)
    wt = rng.uniform(0.1, 2.0, t.shape).astype(np.float32)
    yb, _ = orc.forward(p.astype(np.float64), x.astype(np.float64), bf16=True)
    assert rel(net.forward(x), yb) <= tol_f
    loss, g = net.loss_grad(x, t, wt)
    lb, gb, _ = orc.loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64), bf16=True, wt=wt)
    assert abs(loss - lb) <= 1e-3 * abs(lb)
    for name, (o, shape) in net.layout.items():
        n = int(np.prod(shape))
        assert rel(g[o:o + n], gb[o:o + n]) <= tol_g, name
