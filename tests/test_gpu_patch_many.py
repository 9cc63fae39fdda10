"""A set of more items than one launch can start: a launch counts its work-items in 32 bits, so at 512 lanes to a
workgroup (the sets of short patches, and variants 1 and 3) it holds 2^23 - 1 items and at 1024 lanes (variants 0
and 2) half as many.  8200 patches of 8 x 8 x 512 are 8.4 million items, two or three launches.  Every
patch of the big set must hold, bit by bit, what a set of that patch alone gives (patches at both ends, and those around
the items where launches end)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
COUNT, SHAPE = 8200, (512, 8, 8)     # (nr, nth, nphi): theta and phi take 512 short items each


@pytest.mark.parametrize("variant", [-1, 0, 1, 2, 3])
def test_more_items_than_one_launch_holds(variant):
    from cssx.patches import PatchChunk
    big = PatchChunk([SHAPE] * COUNT, prec="f32")
    gen = torch.Generator(device="cuda").manual_seed(11)
    big.inp.normal_(generator=gen)
    for t in big.out:
        t.fill_(float("nan"))
    print("many patches", variant, flush=True)
    big.run(variant)
    per_patch = {0: 1024 + 1, 1: 1024 + 2, 2: 1024 + 1, 3: 1024 + 2}      # items of a patch, about
    edges = {(1 << 22) // per_patch[0], (1 << 23) // per_patch[1], (1 << 23) // per_patch[0]}
    pick = sorted({0, 1, COUNT - 2, COUNT - 1} | {min(COUNT - 1, e + d) for e in edges for d in (-1, 0, 1)})
    small = PatchChunk([SHAPE] * len(pick), prec="f32")
    for k, i in enumerate(pick):
        small.field(k).copy_(big.field(i))
    small.run(variant)
    for k, i in enumerate(pick):
        for ax in range(3):
            assert torch.equal(small.field(k, ax), big.field(i, ax)), (i, ax)
    for t in big.out:                # (512 x 8 x 8 values, no padding between patches)
        assert torch.isfinite(t).all()
    big.close()
    small.close()
