"""The closure tendency of small grids of whole 16-point tiles.

Time: with at most one tile per wavefront the chip holds (8 to a CU) every tile runs at once, alone in its
wavefront; twice as many tiles take two to a wavefront, whose pass is about 1.6 times as long.  A kernel that always
pairs tiles needs the same time for both grids.  Measured through the FP64 state's call, launch and weight packing
included: 0.77 with single tiles, 0.99 without; the line is 0.88.

Values: a tile's arithmetic does not depend on what else its wavefront does.  The rows of a grid that runs single
tiles must be, bit by bit, those of one that runs pairs and holds the same neighbourhoods."""
import time

import numpy as np
import pytest
import torch

from cssx import closure as cl

pytestmark = pytest.mark.gpu


def _net():
    net = cl.Network(max_rows=64, seed=4)
    rng = np.random.default_rng(9)
    net.set_norm(rng.standard_normal(216) * 1e-3, rng.uniform(5e-3, 2e-2, 216), rng.standard_normal(8) * 1e-2,
                 rng.uniform(0.1, 1.0, 8))
    return net


def _state(shape, dtype):
    gen = torch.Generator(device="cuda").manual_seed(sum(shape))
    return (torch.randn((8,) + shape, dtype=torch.float64, device="cuda", generator=gen) * 1e-2).to(dtype)


def test_one_tile_per_wavefront_where_pairs_leave_compute_units_idle():
    from cssx.model import Config, Model
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    net = _net()
    calls = []
    for nphi in (cus // 8, cus // 4):          # 16 x nphi x 64 points: 8 and 16 tiles per compute unit
        m = Model(Config(nr=16, nth=64, nphi=nphi))
        x = _state((16, nphi, 64), torch.float64)
        out = torch.empty(x.shape, dtype=torch.float32, device="cuda")
        calls.append(lambda x=x, m=m, out=out: cl.tendency(net, x, m, False, out))
    best = [float("inf")] * 2
    for rep in range(30):
        for k, call in enumerate(calls):
            call()
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(50):
                call()
            torch.cuda.synchronize()
            best[k] = min(best[k], time.perf_counter() - t0)
    print("tendency of 8 and 16 tiles per CU:", [b / 50 * 1e6 for b in best], "us", flush=True)
    assert best[0] < 0.88 * best[1]
    net.close()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("tiles_per_row", [1, 17])
def test_single_and_paired_tiles_agree(tiles_per_row, dtype):
    # the first and the last 8 radii of a larger grid in calls of their own: all but the cut radius see the same
    # neighbours.  With 256 CUs the larger grids (2379 and 2295 tiles, odd counts beyond 2048) run pairs, the others
    # single tiles.
    from cssx.model import Config, Model
    nth, nphi = 16 * tiles_per_row, 61 if tiles_per_row == 1 else 9
    big_nr = 39 if tiles_per_row == 1 else 15
    net = _net()
    m = Model(Config(nr=big_nr, nth=nth, nphi=nphi))
    x = _state((big_nr, nphi, nth), dtype)
    big = cl.tendency(net, x, m, True)
    small = cl.tendency(net, x[:, :8].contiguous(), Model(Config(nr=8, nth=nth, nphi=nphi)), True)
    assert torch.equal(big[:, :7], small[:, :7])
    last = cl.tendency(net, x[:, -8:].contiguous(), Model(Config(nr=8, nth=nth, nphi=nphi)), True)
    assert torch.equal(big[:, -7:], last[:, -7:])
    net.close()
