"""How the segmented sweeps of a stage are grouped into launches: blocks of
like pencil length together, the others on their own, against the tiled
sweeps, which take one launch per direction.  Sweeps agree to 1e-13 of the
field maximum (both solve the same pentadiagonal lines, in another order of
operations), whole steps to 1e-12 per conserved variable.  Also the inviscid stage, whose
fluxes are stored before the sweeps."""
import numpy as np
import pytest

from canard_amd import cases
from canard_amd.solver import CanardError, Case, shapes
from helpers import oracle_for, rel_err, tgv_case

pytestmark = pytest.mark.gpu


def _blocks(sizes):
    """Triply periodic blocks, each its own partner, with a perturbed Taylor-Green state."""
    blocks, grids, states = [], [], []
    for i, (lx, ly, lz) in enumerate(sizes):
        blocks.append(dict(lxi=lx, let=ly, lze=lz, nbc=[[45, 45]] * 3, mcd=[[i, i]] * 3))
        grids.append(cases.gridtoy(lx, ly, lz, doml0=0.0, doml1=2 * np.pi, domh=np.pi, span=2 * np.pi))
        states.append(cases.tgv_state(grids[-1], (lx + 1, ly + 1, lz + 1), mach=0.1, pert=1e-3, seed=5 + i))
    return blocks, grids, states, dict(fltk=0.49, fltrbc=0.9, reoo=1.6e4, cfl=0.8, viscous=1)


# more than 512 workgroups of 4 to 16 pencils per class, in two and in four
# classes, the longest pencils first, last and in between; one class whose
# short block has too few pencils
@pytest.mark.parametrize("sizes", [[(40, 92, 90), (150, 92, 90)],
                                   [(99, 90, 66), (290, 40, 66), (150, 68, 64), (31, 92, 91)],
                                   [(120, 60, 60), (30, 20, 18)]])
def test_blocks_of_unlike_length_match_the_tiled_sweeps(sizes):
    blocks, grids, states, params = _blocks(sizes)
    rng = np.random.default_rng(11)
    fields = [np.sin(g[0]) * np.cos(2 * g[1]) + 0.3 * rng.standard_normal(g.shape[1]) for g in grids]
    c = Case(blocks, params)
    c.set_grids(grids)
    c.set_states(states)
    for d in range(3):
        for kind in ("field", "filter"):
            c.set_shape(kind, d, -1)
        want_d, want_f = c.deriv(d, fields), c.filter_sweep(d, fields)
        for sh in [i for i, s in enumerate(shapes()) if s["xi"] == (d == 0)]:
            try:
                c.set_shape("field", d, sh)
                c.set_shape("filter", d, sh)
            except CanardError:   # does not fit these pencils
                continue
            print(f"[classes] {sizes} d={d} shape={sh}", flush=True)
            for got, want in ((c.deriv(d, fields), want_d), (c.filter_sweep(d, fields), want_f)):
                for b in range(len(blocks)):
                    assert np.max(np.abs(got[b] - want[b])) <= 1e-13 * np.max(np.abs(want[b])), (d, sh, b)
    c.close()


@pytest.mark.parametrize("short", [False, True])
def test_steps_of_blocks_of_unlike_length_match_the_tiled_sweeps(short):
    """short: the shapes of few pencils per workgroup, which split into most classes."""
    blocks, grids, states, params = _blocks([(99, 90, 66), (260, 40, 66), (31, 92, 91)])
    out = []
    for tiled in (True, False):
        c = Case(blocks, params)
        c.set_grids(grids)
        c.set_states(states)
        c.set_clock()
        for d in range(3):
            picks = [-1] if tiled else [i for i, s in enumerate(shapes()) if s["xi"] == (d == 0)]
            picks.sort(key=lambda i: shapes()[i]["pencils"] * (1 if short else -1) if i >= 0 else 0)
            for kind in ("filter", "grad", "flux"):
                for sh in picks:
                    try:
                        c.set_shape(kind, d, sh)
                        break
                    except CanardError:
                        continue
        print(f"[classes] steps tiled={tiled} short={short}", flush=True)
        c.step(3)
        out.append([c.state(b) for b in range(len(blocks))])
        c.close()
    for b in range(len(blocks)):
        err = rel_err(out[1][b], out[0][b])
        print("  rel err per variable", err, flush=True)
        assert np.all(err < 1e-12), (b, err)


# stored inviscid fluxes: pointwise kernel, flux sweeps, and the update fused
# into the xi one, its own kernel, or after tiled sweeps
@pytest.mark.parametrize("nxyz", [(12, 13, 16), (40, 36, 34), (67, 33, 20)])
def test_inviscid_steps_match_oracle_fused_separate_and_tiled(monkeypatch, nxyz):
    blocks, grids, states, params = tgv_case(0, nxyz=nxyz, pert=1e-3)
    params["viscous"] = 0
    o = oracle_for(blocks, grids, states, params)
    o.run(5)
    got = {}
    for name, env in (("fused", {}), ("separate", {"CANARD_FUSE_UPDATE": "0"}), ("tiled", {"CANARD_SWEEP": "tiled"})):
        with monkeypatch.context() as m:
            m.setenv("CANARD_TUNE", "0")
            for k, v in env.items():
                m.setenv(k, v)
            print(f"[inviscid] {nxyz} {name}", flush=True)
            c = Case(blocks, params)
        c.set_grids(grids)
        c.set_states(states)
        c.set_clock()
        c.step(5)
        got[name] = c.state(0)
        c.close()
        err = rel_err(got[name], o.state(0))
        print("  rel err per variable", err, flush=True)
        assert np.all(err < 1e-12), (name, err)
    assert np.array_equal(got["fused"], got["separate"])
    o.close()


# pencils of the fewest points (13), of one point more or less than whole
# segments of 9, 17 and 33 points, and between blocks whose partner along d is
# another block (its points staged beside the sweep's own LDS) or themselves
@pytest.mark.parametrize("other", [False, True])
@pytest.mark.parametrize("na,nb", [(13, 18), (19, 27), (28, 17), (34, 67), (101, 55)])
def test_every_shape_at_segment_edges_matches_the_tiled_sweeps(na, nb, other):
    rng = np.random.default_rng(na)
    for d in range(3):
        blocks, fields = [], []
        for i, n in enumerate((na, nb)):
            size = [21, 19, 23]
            size[d] = n
            mcd = [[i, i] for _ in range(3)]
            if other:
                mcd[d] = [1 - i, 1 - i]
            blocks.append(dict(lxi=size[0] - 1, let=size[1] - 1, lze=size[2] - 1, nbc=[[45, 45]] * 3, mcd=mcd))
            fields.append(rng.standard_normal(size[0] * size[1] * size[2]))
        c = Case(blocks, dict(fltk=0.49, fltrbc=0.9))
        for kind in ("field", "filter"):
            c.set_shape(kind, d, -1)
        want_d, want_f = c.deriv(d, fields), c.filter_sweep(d, fields)
        tried = 0
        for sh in [i for i, s in enumerate(shapes()) if s["xi"] == (d == 0)]:
            try:
                c.set_shape("field", d, sh)
                c.set_shape("filter", d, sh)
            except CanardError:   # segments too short or too many
                continue
            tried += 1
            print(f"[edges] {na} {nb} other={other} d={d} shape={sh}", flush=True)
            for got, want in ((c.deriv(d, fields), want_d), (c.filter_sweep(d, fields), want_f)):
                for b in range(2):
                    assert np.max(np.abs(got[b] - want[b])) <= 1e-13 * np.max(np.abs(want[b])), (d, sh, b)
        assert tried > 0
        c.close()


# averaging groups of 2 (one periodic direction), 4 (two) and 8 points (three),
# faces of fewer and more pencils than a workgroup takes, two instances; whole
# steps, whose stages prepare each other, against stages called one by one
@pytest.mark.parametrize("viscous", [1, 0])
@pytest.mark.parametrize("periodic", [(0,), (1,), (2,), (0, 1), (0, 2), (1, 2), (0, 1, 2)])
def test_whole_steps_equal_single_stages_and_oracle(monkeypatch, periodic, viscous):
    monkeypatch.setenv("CANARD_TUNE", "0")   # the same shapes in both
    blocks, grids, states = [], [], []
    for i, (lx, ly, lz) in enumerate([(12, 15, 14), (33, 20, 17)]):
        per = [d in periodic for d in range(3)]
        blocks.append(dict(lxi=lx, let=ly, lze=lz, nbc=[[45, 45] if p else [10, 10] for p in per],
                           mcd=[[i, i] if p else [-1, -1] for p in per], inst=i))
        grids.append(cases.gridtoy(lx, ly, lz, doml0=0.0, doml1=2 * np.pi, domh=np.pi, span=2 * np.pi))
        states.append(cases.tgv_state(grids[-1], (lx + 1, ly + 1, lz + 1), mach=0.1, pert=1e-3, seed=7 + i))
    params = dict(fltk=0.49, fltrbc=0.9, reoo=1.6e4, cfl=0.8, viscous=viscous)
    out = []
    for whole in (True, False):
        print(f"[stages] periodic={periodic} viscous={viscous} whole={whole}", flush=True)
        c = Case(blocks, [params, params])
        c.set_grids(grids)
        c.set_states(states)
        for i in range(2):
            c.set_clock(inst=i)
        if whole:
            c.step(4)
        else:
            for _ in range(4):
                c.filter()
                for nk in range(1, 5):
                    c.rk_stage(nk)
                c.end_step()
        out.append([c.state(b) for b in range(2)])
        c.close()
    for b in range(2):
        assert np.array_equal(out[0][b], out[1][b]), b
        blk = dict(blocks[b], mcd=[[0, 0] if m[0] >= 0 else [-1, -1] for m in blocks[b]["mcd"]])
        o = oracle_for([blk], [grids[b]], [states[b]], params)
        o.run(4)
        err = rel_err(out[0][b], o.state(0))
        print("  rel err per variable", err, flush=True)
        assert np.all(err < 1e-12), (b, err)
        o.close()
