"""compact_fd6 on host arrays without preloaded values: small ones are read and written by the kernel in pinned
host memory and take no darr buffer.  Against the same call with a darr of zeros (copied to the device, plan-driven
kernels), for every boundary code, wall and halo ends, the shortest pencils of each kernel, several
pencils, axes, layouts and types, and both sides of the size line.

Tolerance: both solve the same rows in FP64 (wall rows combine values with coefficient sums near 46 against results of
the order of the inputs): 1e-12 of the largest value."""
import numpy as np
import pytest

from cssx import derivatives
from cssx.derivatives import compact_fd6

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ibc", range(6))
@pytest.mark.parametrize("n", [5, 6, 7, 8, 31, 47, 48, 61, 128, 257, 1024])
def test_no_darr_is_darr_of_zeros(n, ibc):
    rng = np.random.default_rng(n + ibc)
    for dtype in range(4):
        a = rng.standard_normal((n, 3))
        b1, b2 = rng.standard_normal((4, 3)), rng.standard_normal((4, 3))
        want = compact_fd6(1.7 * (n - 1), a, b1, b2, ibc, dtype, np.zeros((n, 3)), axis=0)
        got = compact_fd6(1.7 * (n - 1), a, b1, b2, ibc, dtype, axis=0)
        assert isinstance(got, np.ndarray) and got.shape == a.shape and got.dtype == np.float64
        # (five rows between two Dirichlet-type walls are a singular system: both give the same infinities)
        same = (got == want) | (np.isnan(got) & np.isnan(want))
        assert np.all(np.abs(got - want)[~same] <= 1e-12 * np.abs(want).max()), (n, ibc, dtype)


@pytest.mark.parametrize("shape,axis", [((128,), 0), ((128,), -1), ((9, 64), 1), ((64, 9), 0), ((4, 50, 6), 1),
                                        ((64, 512), 0), ((65, 512), 0), ((512, 64), 1), ((512, 65), 1)])
def test_layouts_and_both_sides_of_the_size_line(shape, axis):
    rng = np.random.default_rng(len(shape) * 100 + axis)
    assert derivatives._HOST_VALUES == 64 * 512
    base = rng.standard_normal(shape)
    z = np.zeros(shape)
    for a in (base, base.astype(np.float32), np.asfortranarray(base), np.repeat(base, 2, axis=-1)[..., ::2], base.tolist()):
        want = compact_fd6(30.0, a, 0.0, 0.0, 1, 0, z.copy(), axis=axis)
        got = compact_fd6(30.0, a, 0.0, 0.0, 1, 0, axis=axis)
        assert got.shape == shape and np.abs(got - want).max() <= 1e-12 * np.abs(want).max()
    for darr in (None, z.copy()):
        with pytest.raises(ValueError):
            compact_fd6(30.0, base[::-1], 0.0, 0.0, 1, 0, darr, axis=axis)
    first = compact_fd6(30.0, base, 0.0, 0.0, 1, 0, axis=axis)
    keep = first.copy()
    compact_fd6(30.0, 2 * base, 0.0, 0.0, 1, 0, axis=axis)      # the staging memory is not the result's
    assert np.array_equal(first, keep)
