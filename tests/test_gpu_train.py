"""The three-launch gradient of the 216-128-128-8 network (csrc/cssx_train.hpp) against the layer-by-layer
path, which serves feature rows that are not 16-byte aligned, at the row counts where it can go wrong: below,
at and past a 32-row workgroup, a 256-row split of the weight gradients, and the most splits.

Both paths round the same values to BF16 and sum the products of a layer in the same order, so their
activations are equal; only the FP32 sums over the rows are ordered differently: at most 8225 terms, whose
rounding stays below 8225 eps = 1e-3 of the sum of magnitudes and is of the order sqrt(8225) eps = 1e-5 of it.
Tolerance: 1e-4 of each block's largest gradient (as for the 8192-term products of test_gpu_closure)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 31, 32, 33, 255, 256, 257, 1000, 8192, 8225])
def test_fused_gradient_matches_the_layer_by_layer_path(rows):
    from cssx import closure as cl
    from oracle import closure as oc
    net = cl.Network(128, 128, max_rows=8225, seed=3)
    g = torch.Generator(device="cuda").manual_seed(rows)
    buf = torch.empty(rows * 216 + 1, dtype=torch.bfloat16, device="cuda")
    x = torch.randn((rows, 216), generator=g, device="cuda").to(torch.bfloat16)
    odd = buf[1:].view(rows, 216)            # two bytes past the allocation: not 16-byte aligned
    odd.copy_(x)
    t = torch.randn((rows, 8), generator=g, device="cuda")
    for step in range(2):
        # the second pass runs on weights that an Adam step wrote (both copies of them)
        loss_f = net.grad(x, t).item()
        gf = net.grads().astype(np.float64)
        loss_l = net.grad(odd, t).item()
        gl = net.grads().astype(np.float64)
        assert abs(loss_f - loss_l) < 1e-5 * loss_l, (rows, loss_f, loss_l)
        for name, a, b in zip(("W1", "b1", "W2", "b2", "W3", "b3"), oc.unpack(gf, 128, 128), oc.unpack(gl, 128, 128)):
            assert np.abs(a - b).max() <= 1e-4 * np.abs(b).max(), (rows, step, name)
        p = net.params()
        loss = net.train_step(x, t, 1e-3).item()
        assert abs(loss - loss_f) < 1e-6 * loss_f
        assert np.abs(net.params() - p).max() > 0
    net.close()
