"""Sweeps of fields that come from memory (over 16 MB in FP32): the segments are then as long as a lane can hold, 20 to 32
rows, where the same lengths of a small field take 16.  One length for each kernel that serves such fields, with
equal segments and with ragged ones, among them 99 rows (five segments of 20 and 19, whose carries span two).

A pencil's derivative depends on that pencil alone: blocks of pencils at the ends and in the middle of the field against
the oracle.  Tolerances as for the small fields: 3e-5 of the largest derivative, 3e-4 where the Dirichlet-type
second derivative's wall pivot is near-singular."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu
LENGTHS = [33, 41, 99, 40, 199, 144, 289, 196, 127, 160, 511, 513, 1024]   # 12 16 20 20= 24 24= 28 28= 32 32= 32, two per wavefront


@pytest.mark.parametrize("n", LENGTHS)
def test_long_segments(n):
    from cssx.operators import Operators
    nth = 131
    other = max(9, -(-4_300_000 // (n * nth)))
    assert other <= 1024 and 4 * n * nth * other > 16e6
    gen = torch.Generator(device="cuda").manual_seed(n)
    for axis, shape in ((0, (n, other, nth)), (2, (other, n, nth))):
        nr, nphi, _ = shape
        d = [1.3 * (nr - 1), 0.7 * (nth - 1), 2.1 * nphi]
        ops = Operators(nr, nth, nphi, *d)
        f = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(generator=gen)
        glo = torch.empty((4, nphi, nth), dtype=torch.float32, device="cuda").normal_(generator=gen) * d[0]
        ghi = torch.empty_like(glo).normal_(generator=gen) * d[0]
        host, hlo, hhi = f.double().cpu().numpy(), glo.double().cpu().numpy(), ghi.double().cpu().numpy()
        for order in (1, 2):
            for bdry in ((0, 1, 2, 3, 4) if axis == 0 else (0,)):
                walls = dict(ghost_lo=glo, ghost_hi=ghi) if axis == 0 else {}
                got = ops.deriv(f, axis, order, bdry, *walls.values()).double().cpu().numpy()
                loose = 10.0 if order == 2 and bdry in (1, 2, 3) else 1.0
                for o in (0, other // 2 - 4, other - 9):
                    for t in (0, 60, nth - 11):
                        at = (slice(None), slice(o, o + 9), slice(t, t + 11)) if axis == 0 else (slice(o, o + 9), slice(None), slice(t, t + 11))
                        g = dict(ghost_lo=np.ascontiguousarray(hlo[at]), ghost_hi=np.ascontiguousarray(hhi[at])) if axis == 0 else {}
                        ref = oracle.deriv_field(axis, order, np.ascontiguousarray(host[at]), lo_wall=axis == 0, hi_wall=axis == 0,
                                                 bdry=bdry, scale=d[axis] ** order, hneu=d[0], **g)
                        err = np.abs(got[at] - ref).max() / np.abs(ref).max()
                        assert err < 3e-5 * loose, (n, axis, order, bdry, o, t, err)
        ops.close()
