"""Elementwise calls over more than 2^32 values, which a launch counts in 32 bits: they are laid out in rows of workgroups."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_features_of_twenty_million_points():
    # 216 features of 320 x 256 x 256 points: 4.5e9 values
    from cssx import closure as cl
    from cssx.model import Config, Model
    nr, nphi, nth = 320, 256, 256
    m = Model(Config(nr=nr, nth=nth, nphi=nphi))
    x = torch.empty((8, nr, nphi, nth), dtype=torch.float32, device="cuda").normal_(generator=torch.Generator(device="cuda").manual_seed(1))
    net = cl.Network(max_rows=64, seed=4)
    rows = nr * nphi * nth
    assert rows * 216 > 1 << 32
    print("features", rows, flush=True)
    every = cl.features(x, m, fluct=True, net=net)
    at = ((1 << 32) // 216)          # the row that a wrapped count would end in
    for row0 in (0, at - 4096 - (1 << 32) // 216 // 2, at - 2048, rows - 4096):
        part = cl.features(x, m, fluct=True, net=net, row0=row0, rows=4096)
        assert torch.equal(every[row0:row0 + 4096], part), row0
    # and standardized in one call
    raw = every.float()
    del every
    std = cl.standardize(raw, np.zeros(216), np.full(216, 2.0), to_bf16=True)
    assert torch.equal(std[-4096:], (raw[-4096:] / 2.0).bfloat16()) and torch.equal(std[at - 2048:at + 2048], (raw[at - 2048:at + 2048] / 2.0).bfloat16())
    net.close()


def test_bound_of_a_large_fp32_state():
    # 8 fields of 540 x 1000 x 1000 points: 4.3e9 values, against the same walls of a small grid
    from cssx.mhd import Solver
    from cssx.model import Config, Model
    ends = [0, 1, -2, -1]
    seen = []
    for nr, nphi, nth in ((9, 10, 11), (540, 1000, 1000)):
        sol = Solver(Model(Config(nr=nr, nth=nth, nphi=nphi)))
        st = torch.ones((8, nr, nphi, nth), dtype=torch.float32, device="cuda")
        print("bound", tuple(st.shape), flush=True)
        sol.bound(st)
        seen.append(st[:, ends][:, :, [0, -1]][:, :, :, ends].clone())
        sol.close()
        del st
    # w on the theta walls, u on the radial ones, the vector potential's two components that the walls hold at zero
    assert (seen[0] == 0).any(dim=3).any(dim=2).any(dim=1).nonzero().flatten().tolist() == [1, 3, 5, 7]
    assert torch.equal(seen[0] == 0, seen[1] == 0)
