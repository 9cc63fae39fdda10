"""r sweeps of FP64 fields of just over 4 GiB, the largest whose pencil rows the kernels reach with 32-bit byte offsets
((nr - 1) planes and one theta row): a workgroup's columns run over the end of a theta row, so that its last
lanes reach further than one theta row.  slack = values to spare: 1 (such a workgroup does not fit), 75
(it does), 566.

A pencil's derivative depends on that pencil alone: sampled blocks of pencils against the oracle, 1e-12 of the
largest derivative as for any FP64 sweep."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr,nth,nphi,slack", [(907, 678, 874, 1), (875, 604, 1017, 75), (877, 605, 1013, 566)])
def test_r_sweep_at_the_offset_limit(nr, nth, nphi, slack):
    from cssx.operators import Operators
    assert (1 << 29) - 1 - nth - (nr - 1) * nth * nphi == slack
    f = torch.empty((nr, nphi, nth), dtype=torch.float64, device="cuda").normal_(generator=torch.Generator(device="cuda").manual_seed(5))
    ops = Operators(nr, nth, nphi, 1.3 * (nr - 1), 1.0, 1.0)
    blocks = [(slice(p, p + 9), slice(t, t + 11)) for p in (0, nphi // 2, nphi - 9) for t in (0, nth // 2, nth - 11)]
    for order in (1, 2):
        print("r sweep", nr, nth, nphi, order, flush=True)
        got = ops.deriv(f, 0, order, 1)
        for p, t in blocks:
            sub = np.ascontiguousarray(f[:, p, t].cpu().numpy())
            ref = oracle.deriv_field(0, order, sub, True, True, 1, scale=(1.3 * (nr - 1)) ** order, hneu=1.3 * (nr - 1))
            err = np.abs(got[:, p, t].cpu().numpy() - ref).max() / np.abs(ref).max()
            assert err < (1e-12 if order == 1 else 1e-11), (order, p, t, err)
        del got
    ops.close()
