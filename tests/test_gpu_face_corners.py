"""Blocks with characteristic faces and walls in all three directions against
the oracle: points in the bands of three faces, whose corrections one lane
applies in order, and corners of three walls, whose conditions the update
applies in order.  The flow runs into all faces and a pressure pulse sits next
to a corner.

Tolerance as for the other step tests with walls: 1e-12 per conserved
variable."""
import numpy as np
import pytest

from canard_amd import cases
from canard_amd.solver import Case
from helpers import oracle_for, rel_err

pytestmark = pytest.mark.gpu

GAM = 1.4


@pytest.mark.parametrize("nbc,viscous", [([[10, 10], [10, 10], [10, 10]], 1), ([[10, 10], [10, 10], [10, 10]], 0),
                                         ([[10, 25], [25, 10], [20, 25]], 1), ([[25, 25], [25, 25], [25, 25]], 1),
                                         ([[20, 20], [20, 20], [20, 20]], 0), ([[20, 10], [25, 20], [10, 20]], 1)])
def test_faces_of_three_directions(nbc, viscous):
    lxi, let, lze = 19, 16, 13
    print(f"[corners] {nbc} viscous={viscous}", flush=True)
    blk = dict(lxi=lxi, let=let, lze=lze, nbc=nbc, mcd=[[-1, -1]] * 3)
    g = cases.gridtoy(lxi, let, lze, doml0=0.0, doml1=float(lxi), domh=let / 2.0, span=float(lze))
    r2 = (g[0] - (lxi - 5.0)) ** 2 + (g[1] - (let / 2.0 - 5.0)) ** 2 + (g[2] - 3.0) ** 2
    p = 1.0 / GAM + 1e-3 / GAM * np.exp(-r2 / 18.0)
    rho = (GAM * p) ** (1.0 / GAM)
    u = (0.1, 0.07, 0.05)
    q = np.stack([rho] + [rho * v for v in u] + [p / (GAM - 1.0) + 0.5 * rho * sum(v * v for v in u)])
    params = dict(reoo=500.0, viscous=viscous, cfl=0.8)
    c = Case([blk], params)
    c.set_grids([g])
    c.set_states([q])
    c.set_clock()
    o = oracle_for([blk], [g], [q], params)
    c.step(25)
    o.run(25)
    got, want = c.state(0), o.state(0)
    assert np.all(np.isfinite(want)) and np.max(np.abs(want - q)) > 1e-3
    err = rel_err(got, want)
    print("  rel err per variable", err, flush=True)
    assert np.all(err < 1e-12), err
    c.close()
    o.close()
