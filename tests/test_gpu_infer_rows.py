"""The closure tendency of grids whose theta rows are whole 16-point tiles, two tiles per wavefront and pass: odd
tile counts (the last wavefront's second tile repeats), fewer tiles than a workgroup takes, pairs that cross
theta rows, phi rows and radii, and more than one pass per wavefront, in both state types, against the
layer-by-layer path.

Bounds as for any two evaluations with the same BF16 rounding points: a hidden activation may round the other way,
2^-8 of one of 128 terms, for a few points in a hundred: 1e-4 of the largest value in the mean, 1e-2 at most."""
import numpy as np
import pytest
import torch

from cssx import closure as cl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(8, 8, 16), (9, 9, 16), (9, 11, 48), (13, 41, 112), (33, 65, 256)])
def test_tendency_of_whole_tiles(shape, prec):
    from cssx.model import Config, Model
    nr, nphi, nth = shape
    m = Model(Config(nr=nr, nth=nth, nphi=nphi))
    rng = np.random.default_rng(nr * nth)
    st = rng.standard_normal((8, nr, nphi, nth)) * 1e-2
    if prec == "f64":
        st[0] += m.rho_bar[:, None, None]
        st[4] += m.s_bar[:, None, None]
    x = torch.as_tensor(st, device="cuda").to(torch.float64 if prec == "f64" else torch.float32).contiguous()
    net = cl.Network(128, 128, max_rows=4096, seed=21)
    xm, xs = rng.standard_normal(216) * 1e-3, rng.uniform(5e-3, 2e-2, 216)
    ym, ys = rng.standard_normal(8) * 1e-2, rng.uniform(0.1, 1.0, 8)
    net.set_norm(xm, xs, ym, ys)
    print("tendency", shape, prec, flush=True)
    got = cl.tendency(net, x, m, fluct=prec == "f32")
    xb = cl.features(x, m, fluct=prec == "f32", net=net)
    pred = torch.cat([net.forward(xb[r:r + 4096].contiguous()) for r in range(0, xb.shape[0], 4096)]).double()
    ref = (pred * torch.as_tensor(ys, device="cuda") + torch.as_tensor(ym, device="cuda")).t().reshape(got.shape)
    d, scale = (got.double() - ref).abs(), ref.abs().max().item()
    assert d.mean().item() < 1e-4 * scale and d.max().item() < 1e-2 * scale, (d.mean().item() / scale, d.max().item() / scale)
    net.close()
