"""The final kernel that solves the theta derivatives itself, in FP32 and at the lengths whose pencils are cut by the
end of a wavefront (two and four wavefronts to a strip, two to four wavefronts to a pencil), with every remainder of the
last lane, tightly enough to see a carry of a hundredth go missing.

Fields of white noise make the theta derivatives as large as the grid allows, so that their rounding is small against
the tendencies they make up; three states keep the seven derivatives from hiding behind one another: velocities
alone (w v u), density and entropy alone, the vector potential alone (B_phi, B_r).  The oracle takes the same
FP32 state.

Tolerance, of each field's largest tendency: a compact derivative of noise is good to 3e-5 of its largest value (250
rounding units, as for the sweeps), a tendency is a sum of up to ten products of such with factors good to a few
rounding units, whose largest value is of the order of the largest term: 3e-4."""
import numpy as np
import pytest
import torch

import oracle
from cssx.model import Config, Model

pytestmark = pytest.mark.gpu
LENGTHS = [33, 34, 35, 36, 129, 130, 131, 132, 169, 170, 171, 172, 257, 258, 259, 260, 386, 387, 388, 389, 513, 514, 515, 516,
           771, 772, 773, 774, 1021, 1022, 1023, 1024]


def noise_states(m, rng):
    """(name, FP64 state) of noise in the velocities, in density and entropy, and in the vector potential."""
    shape = (8, m.c.nr, m.c.nphi, m.c.nth)
    rest = np.zeros(shape)
    rest[0] = m.rho_bar[:, None, None]
    rest[4] = m.s_bar[:, None, None]
    out = []
    for name, fields, amp in (("velocities", (1, 2, 3), 0.1), ("density and entropy", (0, 4), 0.02), ("potential", (5, 6, 7), 0.1)):
        st = rest.copy()
        for f in fields:
            z = amp * rng.uniform(-1.0, 1.0, shape[1:])
            st[f] += z * m.rho_bar[:, None, None] if f == 0 else z
        out.append((name, st))
    return out


def check(m, tol, seed):
    from cssx.mhd import Solver
    sol = Solver(m)
    for name, st in noise_states(m, np.random.default_rng(seed)):
        x = sol.to_f32(torch.as_tensor(st, device="cuda"))
        ref = oracle.rhs(m, sol.from_f32(x).cpu().numpy())
        got = sol.rhs(x).double().cpu().numpy()
        big = np.abs(ref).max(axis=(1, 2, 3))
        err = np.abs(got - ref).max(axis=(1, 2, 3))
        print(name, (m.c.nr, m.c.nth, m.c.nphi), err / np.maximum(big, 1e-30), flush=True)
        # a field that the state leaves alone has no tendency to compare with
        live = big > 1e-3 * big.max()
        assert np.all(err[live] <= tol * big[live]), (name, err, big)
    sol.close()


@pytest.mark.parametrize("nth", LENGTHS)
def test_noise_over_theta_lengths(nth):
    check(Model(Config(nr=9, nth=nth, nphi=10)), 3e-4, nth)


@pytest.mark.parametrize("nr,nth,nphi", [(64, 20, 72), (61, 21, 67), (128, 20, 49), (33, 9, 127)])
def test_noise_with_short_segments(nr, nth, nphi):
    # the batched sweeps of small fields along r and phi (8-row segments), FP32, and FP64 against the oracle
    from cssx.mhd import Solver
    m = Model(Config(nr=nr, nth=nth, nphi=nphi))
    check(m, 3e-4, nr)
    sol = Solver(m)
    for name, st in noise_states(m, np.random.default_rng(nphi)):
        ref = oracle.rhs(m, st)
        err = np.abs(sol.rhs(torch.as_tensor(st, device="cuda")).cpu().numpy() - ref).max(axis=(1, 2, 3))
        big = np.abs(ref).max(axis=(1, 2, 3))
        assert np.all(err <= 1e-10 * np.maximum(big, big.max() * 1e-6)), (name, err, big)
    sol.close()


def test_very_large_field_with_a_ragged_theta_axis():
    """From 400 MB a field on the kernel's workgroups are dealt out in another order, and the last of them, whose last lane
    may reach past the fields, is told apart by its place: 400 x 1000 x 251 in FP32 (402 MB) against FP64, whose
    ragged lengths keep the sweeps and the pointwise final kernel.  A workgroup out of place misses by the tendency
    itself; 1e-3 of it covers FP32."""
    from cssx.mhd import Solver
    nr, nphi, nth = 400, 1000, 251
    m = Model(Config(nr=nr, nth=nth, nphi=nphi))
    sol = Solver(m)
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.empty((8, nr, nphi, nth), dtype=torch.float32, device="cuda").uniform_(-0.1, 0.1, generator=gen)
    x[0] *= torch.as_tensor(m.rho_bar, dtype=torch.float32, device="cuda")[:, None, None] * 0.2
    x[4] *= 0.2
    got = sol.rhs(x)
    ref = sol.rhs(sol.from_f32(x))
    for f in range(8):
        big = ref[f].abs().max().item()
        err = max((got[f, r].double() - ref[f, r]).abs().max().item() for r in range(nr))
        print("large ragged", f, err / big, flush=True)
        assert err <= 1e-3 * big, (f, err, big)
    sol.close()
