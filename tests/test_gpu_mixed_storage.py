"""What mixed precision changes, and by how much: the eta and zeta gradients of
viscous stages are stored in FP32 and nothing else, so the sweeps and inviscid
steps are bit for bit those of FP64 (the shapes are the default ones in both),
and a viscous step differs by the rounding of those gradients only.

Bound of that difference: a gradient g is stored with an error of at most
2^-24 |g|.  A stress row adds at most 3 of them times the viscosity 1 / Re, a
heat flux about 3.5 (gamma - 1)^-1 Pr^-1 more, so a flux is off by at most
2^-24 12 G / Re with G the largest gradient; differentiating that along
direction d of spacing h_d gives at most 2.4 / h_d of it (the compact scheme's
largest modified wavenumber), and a run of length t adds at most t times the
sum over the directions.  Blocks whose eta and zeta sweeps share a launch and
blocks whose do not, and two blocks with another as partner."""
import numpy as np
import pytest

from canard_amd import cases
from canard_amd.solver import CND_FP64, CND_MIXED, Case
from helpers import tgv_case

pytestmark = pytest.mark.gpu

GAM = 1.4


def _tgv(nxyz):
    blocks, grids, states, params = tgv_case(0, nxyz=nxyz, pert=1e-3)
    h = [2 * np.pi / n for n in nxyz]
    return blocks, grids, states, dict(params, reoo=200.0), 200.0, h


def _pair():
    sizes = [(20, 26, 14), (17, 26, 14)]
    grids = cases.sheared_pair_grids(sizes, h=1.0, amp=0.05)
    states = [cases.pulse_state(g, mach=0.3, centres=[(14.0, 8.0, 6.0)], amp=1e-2, width=3.0) for g in grids]
    # (the shear, x = X + 0.05 Lx sin(2 pi Y / Ly), lengthens eta's lines and shortens none)
    return cases.sheared_pair_blocks(sizes), grids, states, dict(reoo=30.0, amach1=0.3, nsmf=1, cfl=0.8), 100.0, [1.0] * 3


CASES = {"joint 45x41x37": lambda: _tgv((44, 40, 36)), "apart 31x21x71": lambda: _tgv((30, 20, 70)), "pair": _pair}


def _gradient(blocks, states, h):
    """Largest difference of neighbouring points' u, v, w, T over the spacing."""
    G = 0.0
    for b, q in zip(blocks, states):
        u = q[1:4] / q[0]
        T = GAM * (GAM - 1) * (q[4] - 0.5 * q[0] * np.sum(u * u, axis=0)) / q[0]
        f = np.concatenate([u, T[None]]).reshape(4, b["lze"] + 1, b["let"] + 1, b["lxi"] + 1)
        G = max([G] + [float(np.max(np.abs(np.diff(f, axis=3 - d)))) / h[d] for d in range(3)])
    return G


def _run(blocks, grids, states, params, precision, steps):
    c = Case(blocks, params, precision=precision)
    c.set_grids(grids)
    c.set_states(states)
    c.set_clock()
    c.step(steps)
    return c


@pytest.mark.parametrize("name", CASES)
def test_sweeps_and_inviscid_steps_are_those_of_fp64(monkeypatch, name):
    monkeypatch.setenv("CANARD_TUNE", "0")
    blocks, grids, states, params, _, _ = CASES[name]()
    print(f"[mixed storage] {name} inviscid", flush=True)
    a, b = (_run(blocks, grids, states, dict(params, viscous=0), p, 8) for p in (CND_FP64, CND_MIXED))
    fields = [q[1] for q in states]
    for d in range(3):
        for k in range(len(blocks)):
            assert np.array_equal(a.deriv(d, fields)[k], b.deriv(d, fields)[k])
            assert np.array_equal(a.filter_sweep(d, fields)[k], b.filter_sweep(d, fields)[k])
    for k in range(len(blocks)):
        assert np.array_equal(a.state(k), b.state(k))
    a.close()
    b.close()


@pytest.mark.parametrize("name", CASES)
def test_viscous_steps_differ_by_the_rounding_of_the_gradients(monkeypatch, name):
    monkeypatch.setenv("CANARD_TUNE", "0")
    blocks, grids, states, params, re, h = CASES[name]()
    print(f"[mixed storage] {name} viscous", flush=True)
    a, b = (_run(blocks, grids, states, dict(params, viscous=1), p, 20) for p in (CND_FP64, CND_MIXED))
    G = _gradient(blocks, states, h)
    bound = 2.0 ** -24 * 12.0 * G / re * sum(2.4 / v for v in h) * a.clock()["timo"]
    diff = max(float(np.max(np.abs(a.state(k) - b.state(k)))) for k in range(len(blocks)))
    print(f"  difference {diff:.2e}, bound {bound:.2e}, largest gradient {G:.3f}", flush=True)
    assert 0.0 < diff <= bound
    a.close()
    b.close()
