"""The variant that a set of patches starts with.  Axes too short for the constant-coefficient items run on plan-driven
ones, which cover the pencils of one plane and leave most of a large workgroup's lanes idle: sets made of them start with
512-lane workgroups.  The start must not be far behind the best of the four variants (1024 lanes: 2.2 to 2.5 times on
these sets; the line is 1.5)."""
import time

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("name", ["16^3", "8..31", "flat", "32..256"])
def test_the_start_is_near_the_best_variant(name, prec):
    from cssx.patches import PatchChunk
    rng = np.random.default_rng(3)
    shapes = {"16^3": [(16, 16, 16)] * 256, "8..31": rng.integers(8, 32, (64, 3)),
              "flat": [(512, 8, 8), (8, 512, 8), (8, 8, 512)] * 20, "32..256": rng.integers(32, 257, (24, 3))}[name]
    ch = PatchChunk(shapes, prec=prec)
    ch.inp.normal_()
    best = {}
    for rep in range(12):
        for variant in (-1, 0, 1, 2, 3):
            ch.run(variant)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(10):
                ch.run(variant)
            torch.cuda.synchronize()
            best[variant] = min(best.get(variant, float("inf")), time.perf_counter() - t0)
    print(name, prec, {v: round(t * 1e5, 1) for v, t in best.items()}, "us", flush=True)
    assert best[-1] < 1.5 * min(best.values())
    ch.close()
