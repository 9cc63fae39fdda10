"""SLD with the field but without Magnetic_Diffusion: the vector potential has no SLD tendency.  cssx_diffusion must say so
in its output (here handed over full of NaN), and the steps must not add what their scratch memory held before: device
memory full of NaN is given back right before the solver takes its own.  Tolerances as in test_gpu_sld: 1e-11 and 1e-4 of each field's largest
tendency, 1e-9 and 1e-3 of its largest change."""
import numpy as np
import pytest
import torch

import oracle
from cssx.model import Config, Model

pytestmark = pytest.mark.gpu
SHAPE = dict(nr=20, nth=48, nphi=24)


def _setup(**kw):
    from cssx.mhd import Solver
    m = Model(Config(**SHAPE, sld_coef=0.3, Magnetic_Diffusion=False, **kw))
    st = m.initial_state()
    R, P, T = np.meshgrid(m.r, m.phi, m.theta, indexing="ij")
    st[1] += 1e-2 * np.sin(3 * R) * np.sin(2 * T) * np.cos(2 * P)
    st[2] += 1e-2 * np.cos(2 * R) * np.sin(T) * np.sin(2 * P + 0.3)
    st[3] += 1e-2 * np.sin(5 * R) * np.sin(3 * T) * np.cos(2 * P + 1.0)
    st = oracle.bound(m, st)
    torch.cuda.empty_cache()
    stale = [torch.full((n,), float("nan"), dtype=torch.float64, device="cuda") for n in (20 * 48 * 24 * 8, 1 << 20, 1 << 24, 1 << 26)]
    torch.cuda.synchronize()
    del stale
    torch.cuda.empty_cache()
    return m, Solver(m), st


@pytest.mark.parametrize("heating", [True, False])
def test_diffusion_leaves_the_vector_potential_alone(heating):
    m, sol, st = _setup(Do_Ohmic_Heating=heating)
    ref = oracle.diffusion(m, st)
    assert np.all(ref[5:] == 0)
    x = torch.as_tensor(st, device="cuda")
    for z, tol in ((x, 1e-11), (sol.to_f32(x), 1e-4)):
        got = sol.diffusion(z, out=torch.full_like(z, float("nan"))).double().cpu().numpy()
        assert np.all(got[5:] == 0)
        err = np.abs(got - ref).max(axis=(1, 2, 3))[:5]
        assert np.all(err <= tol * np.abs(ref).max(axis=(1, 2, 3))[:5]), err
    sol.close()


@pytest.mark.parametrize("scheme", ["rk4", "rk3_tvd", "rk2_tvd"])
def test_steps_add_nothing_to_it(scheme):
    m, sol, st = _setup()
    ref = oracle.rk4(m, st, 2e-5, 2, scheme=scheme)
    d0 = np.abs(ref - st).max(axis=(1, 2, 3))
    for prec, tol in (("f64", 1e-9), ("f32", 1e-3)):
        print(scheme, prec, flush=True)
        y = torch.as_tensor(st, device="cuda").contiguous()
        sol.rk4(y, 2e-5, 2, prec, scheme)
        err = np.abs(y.cpu().numpy() - ref).max(axis=(1, 2, 3))
        assert np.all(err <= tol * d0 + 1e-15), (err, d0)
    sol.close()
