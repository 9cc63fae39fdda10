"""Patches whose axis lengths sit at the edges of the batched kernel's item kinds: the last plan-driven and the
first constant-coefficient lengths (31 / 32 in FP32, 47 / 48 in FP64), the power-of-two segment counts and their
shortest segments, and partial last lanes, against the oracle in every variant.  Tolerances as in
test_gpu_patches: FP64 1e-12 and FP32 3e-5 of the largest derivative."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu
SHAPES = [(31, 32, 33), (47, 48, 49), (64, 65, 66), (97, 15, 128), (129, 130, 9), (256, 10, 257), (10, 511, 13),
          (11, 258, 385), (513 - 1, 33, 8)]


@pytest.mark.parametrize("bdry", [1, 2])
@pytest.mark.parametrize("prec,tol", [("f64", 1e-12), ("f32", 3e-5)])
def test_item_kinds_match_the_oracle(prec, tol, bdry):
    from cssx.patches import PatchChunk
    ch = PatchChunk(SHAPES, prec=prec, bdry=bdry)
    rng = np.random.default_rng(7 + bdry)
    refs = []
    for i, (nr, nth, nphi) in enumerate(SHAPES):
        ch.field(i).copy_(torch.as_tensor(rng.standard_normal((nr, nphi, nth))))
        f = ch.field(i).double().cpu().numpy()
        g = np.ascontiguousarray(f.transpose(1, 0, 2))   # phi as the slow axis: the r operator with walls
        refs.append((oracle.deriv_field(0, 1, f, True, True, bdry, scale=nr - 1, hneu=nr - 1),
                     oracle.deriv_field(1, 1, f, True, True, bdry, scale=nth - 1, hneu=nth - 1),
                     oracle.deriv_field(0, 1, g, True, True, bdry, scale=nphi - 1, hneu=nphi - 1).transpose(1, 0, 2)))
    for variant in range(4):
        for t in ch.out:
            t.fill_(float("nan"))
        ch.run(variant)
        for i in range(len(SHAPES)):
            for ax in range(3):
                got = ch.field(i, ax).double().cpu().numpy()
                err = np.abs(got - refs[i][ax]).max() / np.abs(refs[i][ax]).max()
                assert err < tol, (variant, SHAPES[i], ax, err)
    ch.close()
