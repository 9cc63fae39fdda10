"""The final kernel that solves the theta derivatives itself (4 rows per lane, from 48 rows in FP64 and 32 in FP32 on)
against the oracle, at the theta lengths where its lane layout changes: the shortest it takes, every
remainder of the last lane, one and several pencils per wavefront, pencils cut by a wavefront's end (two and
four wavefronts to a strip), and the longest.  9 x 10 pencils, no multiple of any strip's.

Tolerances.  FP64: 1e-10 of each field's largest tendency (the entropy's is 1e-2 of s, so its rounding there
is near 1e-11).  FP32: the derivative of O(1) fields rounds at eps32 * 2 dti, against tendencies as
small as 1e-2: 1.2e-5 dti, taken five times.  A step: 1e-9 and 1e-3 of each field's largest change."""
import numpy as np
import pytest
import torch

import mms
import oracle
from cssx.model import Config, Model

pytestmark = pytest.mark.gpu
LENGTHS = [32, 33, 47, 48, 49, 50, 51, 64, 65, 96, 97, 129, 151, 193, 255, 256, 257, 258, 259, 260, 386, 512, 513, 771, 1021, 1024]


def _rel(a, b):
    return np.array([np.abs(a[i] - b[i]).max() / max(np.abs(b[i]).max(), 1e-300) for i in range(a.shape[0])])


HYDRO = [n for n in LENGTHS if n % 4 == 0] + [33, 50, 259]


@pytest.mark.parametrize("nth,magnetic", [(n, True) for n in LENGTHS] + [(n, False) for n in HYDRO])
def test_rhs_over_theta_lengths(nth, magnetic):
    from cssx.mhd import Solver
    m = Model(Config(nr=9, nth=nth, nphi=10, omega0=0.3, damping_time=50.0, magnetic=magnetic))
    st = mms.evaluate(Model(Config(nr=9, nth=nth, nphi=10, omega0=0.3, damping_time=50.0)))[0][:8 if magnetic else 5]
    ref = oracle.rhs(m, st)
    sol = Solver(m)
    x = torch.as_tensor(np.ascontiguousarray(st), device="cuda")
    print("rhs", nth, magnetic, flush=True)
    e = _rel(sol.rhs(x).cpu().numpy(), ref)
    assert e.max() < 1e-10, e
    e32 = _rel(sol.rhs(sol.to_f32(x)).double().cpu().numpy(), ref)
    assert e32.max() < max(5e-3, 6e-5 * m.dti), e32
    sol.close()


@pytest.mark.parametrize("sld", [True, False])
@pytest.mark.parametrize("nth", [50, 97, 256, 259])
def test_step_over_theta_lengths(nth, sld):
    from cssx.mhd import Solver
    m = Model(Config(nr=9, nth=nth, nphi=10, omega0=0.3, **(dict(sld_coef=0.3) if sld else {})))
    st = m.initial_state()
    R, P, T = np.meshgrid(m.r, m.phi, m.theta, indexing="ij")
    st[1] += 1e-2 * np.sin(3 * R) * np.sin(2 * T) * np.cos(2 * P)
    st[2] += 1e-2 * np.cos(2 * R) * np.sin(T) * np.sin(2 * P + 0.3)
    st[3] += 1e-2 * np.sin(5 * R) * np.sin(3 * T) * np.cos(2 * P + 1.0)
    st = oracle.bound(m, st)
    dt = 2e-5
    ref = oracle.rk4(m, st, dt, 2)
    d0 = np.abs(ref - st).max(axis=(1, 2, 3))
    sol = Solver(m)
    for prec, tol in (("f64", 1e-9), ("f32", 1e-3)):
        print("step", nth, sld, prec, flush=True)
        y = torch.as_tensor(st, device="cuda").contiguous()
        sol.rk4(y, dt, 2, prec)
        chg = np.abs(y.cpu().numpy() - ref).max(axis=(1, 2, 3))
        assert np.all(chg <= tol * d0 + 1e-15), (chg, d0)
    sol.close()
