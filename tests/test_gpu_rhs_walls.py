"""The wall kernels of the right-hand side and the density's radial derivative from a sweep with zero wall values
plus the walls' response, against the oracle: radii from the fewest to several segments of the r sweep (on the
plan-driven and the constant-coefficient kernels); and the Compute_B wall conditions, exactly: zero where a wall's
condition says so, for every pair of conditions, and nowhere else.

Tolerances of the first.  FP64: 1e-10 of each field's largest tendency.  FP32: the derivative of O(1) fields rounds at
eps32 * 2 / (cell width), against tendencies as small as 1e-2: 1.2e-5 / width, taken five times."""
import numpy as np
import pytest
import torch

import mms
import oracle
from cssx.model import Config, Model

pytestmark = pytest.mark.gpu

SHUT = dict(Top_Radial_Field=False, Bottom_Radial_Field=False, Top_Perfect_Cond=True, Bottom_Perfect_Cond=True)
CONDUCTOR = dict(Theta_Normal_Field=False, Theta_Perf_Conductor=True)
WALLS = {"normal_radial": {}, "conductor_radial": CONDUCTOR, "normal_shut": SHUT, "conductor_shut": {**SHUT, **CONDUCTOR}}


def _check(cfg):
    from cssx.mhd import Solver
    m = Model(Config(**cfg))
    st = mms.evaluate(Model(Config(nr=cfg["nr"], nth=cfg["nth"], nphi=cfg["nphi"])))[0]
    ref = oracle.rhs(m, st)
    sol = Solver(m)
    x = torch.as_tensor(np.ascontiguousarray(st), device="cuda")
    top = np.abs(ref).reshape(8, -1).max(axis=1)
    e = np.abs(sol.rhs(x).cpu().numpy() - ref).reshape(8, -1).max(axis=1) / top
    assert e.max() < 1e-10, e
    width = 1.0 / max(m.dti, m.dri * float(np.abs(m.dxdr).max()))
    e32 = np.abs(sol.rhs(sol.to_f32(x)).double().cpu().numpy() - ref).reshape(8, -1).max(axis=1) / top
    sol.close()
    return e32.max(), max(5e-3, 6e-5 / width)


@pytest.mark.parametrize("nr", [8, 9, 16, 31, 32, 33, 48, 65])
def test_rhs_over_radii(nr):
    print("radii", nr, flush=True)
    got, tol = _check(dict(nr=nr, nth=49, nphi=11))
    assert got < tol, (got, tol)


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("walls", sorted(WALLS))
def test_b_on_the_walls(walls, precision):
    from cssx.mhd import Solver
    m = Model(Config(nr=9, nth=34, nphi=12, **WALLS[walls]))
    st = torch.as_tensor(np.random.default_rng(3).standard_normal((8, 9, 12, 34)) * 1e-2, device="cuda")
    st[0] += 1.0
    sol = Solver(m)
    print("b walls", walls, precision, flush=True)
    _, b = sol.rhs(st if precision == "f64" else sol.to_f32(st), want_b=True)
    zero = torch.zeros((3, 9, 12, 34), dtype=torch.bool)
    for comp in ([0] if m.c.Theta_Perf_Conductor else [1, 2]):
        zero[comp, :, :, [0, -1]] = True
    if m.c.Bottom_Radial_Field:
        zero[:2, 0] = True
    if m.c.Top_Radial_Field:
        zero[:2, -1] = True
    assert torch.equal((b == 0).cpu(), zero)
    sol.close()
