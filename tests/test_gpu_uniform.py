"""Sweeps of pencils long enough for the constant-coefficient kernels (walls at both ends or the periodic
wrap, from 48 rows in FP64 and 32 in FP32 on) against the oracle, at the lengths where their segmentation
changes: the first ones they take, partial last lanes (n mod 8), one and two segments per wavefront, and
the largest.  Pencil counts are no multiple of a wavefront's columns.

Tolerance.  Relative to the largest derivative, white noise: a solution is a sum of right-hand sides with
geometric weights (sum 1/(p (1-a)^2) < 3.1), its wall rows combine values with coefficient sums near 46
(first derivative) or 80 and, for a Dirichlet-type second derivative, divide by the eliminated wall pivot
0.012, all against results of the order of the inputs; 1e-12 and 3e-5 are 4500 and 250 rounding units, and
1e-11 and 3e-4 for the near-singular pivot."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu
LENGTHS = [31, 32, 33, 40, 47, 48, 49, 50, 56, 57, 63, 64, 65, 97, 128, 129, 192, 255, 256, 257, 273, 511, 512, 513, 529,
           1023, 1024]


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("n", LENGTHS)
def test_sweeps_match_the_oracle(n, order):
    import sys, os
    sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "css-code_amd"))
    from cssx.operators import Operators
    rng = np.random.default_rng(n * 10 + order)
    for axis in (0, 1, 2):
        shape = [(n, 9, 11), (9, 11, n), (9, n, 11)][axis]
        nr, nphi, nth = shape
        f = rng.standard_normal(shape)
        dri, dti, dpi = 1.3 * (nr - 1), 0.7 * (nth - 1), 2.1 * nphi
        ops = Operators(nr, nth, nphi, dri, dti, dpi)
        d = [dri, dti, dpi][axis]
        # ghost buffers carry the prescribed wall derivative in slot 0
        gshape = [(4, nphi, nth), (nr, nphi, 4), None][axis]
        for bdry in ((0, 1, 2, 3, 4) if axis < 2 else (0,)):
            glo = ghi = None
            if axis < 2:
                glo, ghi = rng.standard_normal(gshape) * d, rng.standard_normal(gshape) * d
            ref = oracle.deriv_field(axis, order, f, lo_wall=axis < 2, hi_wall=axis < 2, bdry=bdry, ghost_lo=glo,
                                     ghost_hi=ghi, scale=d if order == 1 else d * d, hneu=d if order == 1 else dri)
            loose = 10.0 if order == 2 and bdry in (1, 2, 3) else 1.0
            for prec, tol in ((torch.float64, 1e-12), (torch.float32, 3e-5)):
                t = lambda x: None if x is None else torch.as_tensor(x, dtype=prec, device="cuda")  # noqa: E731
                got = ops.deriv(t(f), axis, order, bdry, t(glo), t(ghi)).double().cpu().numpy()
                err = np.abs(got - ref).max() / np.abs(ref).max()
                assert err < tol * loose, (n, axis, order, bdry, prec, err)
        ops.close()
