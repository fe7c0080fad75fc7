"""Inviscid flux sweeps where some directions take the tiled sweep, which
evaluates the fluxes from the state, and the others the segmented one, which
reads stored fluxes: every combination of directions against the oracle, on
two blocks that are each other's partner along xi, and a block whose xi
pencils are too long for the segmented sweeps.  Nothing is stored for a
direction that does not read it: with three tiled directions the stage has no
flux kernel, as it had before segmented sweeps took theirs stored.

Tolerance as for the other step tests: 1e-12 per conserved variable."""
import numpy as np
import pytest

from canard_amd import cases
from canard_amd.solver import Case
from helpers import oracle_for, rel_err, tgv_case

pytestmark = pytest.mark.gpu

STEPS = 4


def _pair():
    """Two blocks periodic through each other along xi, each its own partner along eta and zeta."""
    n0, n1, let, lze = 21, 17, 18, 15
    h = 2 * np.pi / (n0 + n1)
    blocks = [dict(lxi=n, let=let, lze=lze, nbc=[[45, 35] if b == 0 else [35, 45], [45, 45], [45, 45]],
                   mcd=[[1 - b, 1 - b], [b, b], [b, b]]) for b, n in enumerate((n0, n1))]
    grids = [cases.gridtoy(n0, let, lze, doml0=0.0, doml1=n0 * h, domh=np.pi, span=2 * np.pi),
             cases.gridtoy(n1, let, lze, doml0=-n0 * h, doml1=(n0 + n1) * h, domh=np.pi, span=2 * np.pi)]
    states = [cases.tgv_state(g, (b["lxi"] + 1, let + 1, lze + 1), mach=0.1) for g, b in zip(grids, blocks)]
    return blocks, grids, states, dict(fltk=0.49, fltrbc=0.9, reoo=1.6e4, cfl=0.8)


def _run(blocks, grids, states, params, tiled):
    c = Case(blocks, params)
    c.set_grids(grids)
    c.set_states(states)
    c.set_clock()
    for d in tiled:
        c.set_shape("flux", d, -1)
    c.profile(True)
    c.step(STEPS)
    return c, c.profile_read()["stress"][1]


@pytest.mark.parametrize("tiled", [(), (0,), (1,), (2,), (0, 1), (0, 2), (1, 2), (0, 1, 2)])
def test_inviscid_steps_with_some_directions_tiled(monkeypatch, tiled):
    monkeypatch.setenv("CANARD_TUNE", "0")
    blocks, grids, states, params = _pair()
    params["viscous"] = 0
    print(f"[tiled flux] {tiled}", flush=True)
    o = oracle_for(blocks, grids, states, params)
    o.run(STEPS)
    c, stored = _run(blocks, grids, states, params, tiled)
    for b in range(2):
        err = rel_err(c.state(b), o.state(b))
        print("  rel err per variable", err, flush=True)
        assert np.all(err < 1e-12), (tiled, b, err)
    assert stored == (0 if len(tiled) == 3 else 4 * STEPS)
    c.close()
    o.close()


@pytest.mark.parametrize("viscous", [0, 1])
def test_pencils_too_long_for_segments(viscous):
    blocks, grids, states, params = tgv_case(0, nxyz=(530, 13, 14), pert=1e-3)
    params["viscous"] = viscous
    print(f"[tiled flux] 531 points, viscous={viscous}", flush=True)
    o = oracle_for(blocks, grids, states, params)
    o.run(STEPS)
    c, _ = _run(blocks, grids, states, params, ())
    assert c.tuning()["flux"][0]["shape"] == -1
    err = rel_err(c.state(0), o.state(0))
    print("  rel err per variable", err, flush=True)
    assert np.all(err < 1e-12), err
    c.close()
    o.close()
