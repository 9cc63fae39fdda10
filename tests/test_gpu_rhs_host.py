"""Host time of a right-hand side: what depends on sizes and flags alone is worked out when the solver is made.  The
lane layout of the final kernel is a search over wavefronts, pencils and offsets that takes longest at the shortest
theta pencils (30 us at 32 rows, under 2 at 512); the calls of both lengths make the same launches, so handing them over
must cost the same.  The line, 1.25, lies between 1.0 and the 1.6 or more of a search in every call."""
import time

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_short_pencils_cost_the_host_no_more_than_long_ones():
    from cssx.mhd import Solver
    from cssx.model import Config, Model
    calls, keep = [], []
    for nth in (32, 512):
        m = Model(Config(nr=8, nth=nth, nphi=8))
        sol = Solver(m)
        x = sol.to_f32(torch.as_tensor(m.initial_state(), device="cuda").contiguous())
        out = torch.empty_like(x)
        keep.append((sol, x, out))
        calls.append(lambda sol=sol, x=x, out=out: sol.rhs(x, out))
    best = [float("inf")] * 2
    for rep in range(60):
        for k, call in enumerate(calls):
            call()
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(8):
                call()
            best[k] = min(best[k], time.perf_counter() - t0)   # (handed over, not finished)
            torch.cuda.synchronize()
    print("right-hand side, host us at 32 and 512 rows:", [b / 8 * 1e6 for b in best], flush=True)
    assert best[0] < 1.25 * best[1]
    for sol, _, _ in keep:
        sol.close()
