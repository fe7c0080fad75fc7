"""Performance cases: what users of canard_amd have it do, through `Case` and `Net`.

A pass is a piece of a run as a solver user drives it: a number of whole time steps, then the state (and the
clock, and the recorded averages where the run records) is read back, as a program does between two outputs.  Only
the read-back waits for the device.  Closure users train the network on stored pairs, or run a coarse block with
the network's correction after every step.

Sizes are those of this repository's configurations, tests and benchmark; `draw` spreads the same kinds over the
ranges in between, odd and uneven sizes included.  All inputs come from the seed: a Taylor-Green vortex with random
resolved modes and grid-scale noise, pressure pulses in a Mach 0.5 stream, or normalised flow fields with small
corrections for the network.

`exact` restates the periodic step and the network in 64 bits with plain numpy and torch: a compact derivative or
filter along one direction is a dense matrix there.
"""
import math

import numpy as np
import torch

from canard_amd import cases as setup
from canard_amd.closure import Net
from canard_amd.solver import CND_FP64, CND_MIXED, Case

GAM, PRANDTL = 1.4, 0.71
FLTK, FLTRBC, TEMPOO, CFL = 0.49, 0.9, 300.0, 0.8
PARAMS = dict(fltk=FLTK, fltrbc=FLTRBC, tempoo=TEMPOO, cfl=CFL)
CHANNELS = (5, 32, 32, 5)   # the closure network: three 3x3x3 convolutions


def listed():
    return [
        # the smallest block in use (a smoke run): a step is a few dozen short dependent launches
        dict(name="tgv_16", kind="periodic", nx=16, ny=16, nz=16, viscous=True, mixed=False, graph=False, steps=20),
        # the 64^3 vortex of 100 steps, replayed as a graph: ordinary resolution, latency and bandwidth both count
        dict(name="tgv_64_graph", kind="periodic", nx=64, ny=64, nz=64, viscous=True, mixed=False, graph=True, steps=100),
        # the benchmark's block, launched kernel by kernel: every sweep streams from HBM
        dict(name="tgv_256", kind="periodic", nx=256, ny=256, nz=256, viscous=True, mixed=False, graph=False, steps=40),
        # the same flow in mixed precision at the middle size of the configurations
        dict(name="tgv_128_mixed", kind="periodic", nx=128, ny=128, nz=128, viscous=True, mixed=True, graph=False, steps=40),
        # an uneven inviscid box: fluxes come straight from the state, directions differ in length
        dict(name="euler_100x60x40", kind="periodic", nx=100, ny=60, nz=40, viscous=False, mixed=False, graph=False, steps=40),
        # a channel with an inviscid and an isothermal wall and non-reflective ends, recording time averages
        dict(name="channel_80x70x50", kind="channel", nx=80, ny=70, nz=50, steps=40),
        # four uneven sheared blocks with characteristic faces, interfaces and a sponge, 15 M points
        dict(name="sheared_blocks", kind="sheared", nx=384, nx2=192, ny=256, nz=64, steps=30),
        # a parameter study: many small vortices of two sizes batched in one context, replayed as a graph
        dict(name="ensemble_32", kind="ensemble", count=32, lo=24, hi=32, steps=50),
        # training the closure at the size the 64^3 coarse runs use, and on a smaller coarse grid
        dict(name="train_64", kind="train", n=64, pairs=4, iters=20),
        dict(name="train_32", kind="train", n=32, pairs=4, iters=20),
        # a coarse run with the trained network's correction after every step
        dict(name="closure_run_64", kind="apply", n=64, steps=20),
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _steps(rng, points):
    """10 to 60 steps, within 40 steps of the largest block."""
    return max(4, min(rng.randint(10, 60), int(40 * 257 ** 3 / points)))


def draw(rng):
    kind = rng.choice(["periodic"] * 5 + ["channel", "sheared", "ensemble", "train", "apply"])
    if kind == "periodic":
        nx, ny, nz = (_size(rng, 12, 180) for _ in range(3))
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, viscous=rng.random() < 0.75, mixed=rng.random() < 0.25,
                    graph=rng.random() < 0.4, steps=_steps(rng, nx * ny * nz))
    if kind == "channel":
        nx, ny, nz = (_size(rng, 16, 120) for _ in range(3))
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, steps=_steps(rng, nx * ny * nz))
    if kind == "sheared":
        nx, nx2, ny, nz = (_size(rng, 24, hi) for hi in (260, 180, 160, 60))
        return dict(kind=kind, nx=nx, nx2=nx2, ny=ny, nz=nz, steps=_steps(rng, 2 * (nx + nx2) * ny * nz))
    if kind == "ensemble":
        lo = _size(rng, 12, 48)
        hi, count = lo + rng.randint(1, 24), rng.randint(6, 32)
        return dict(kind=kind, count=count, lo=lo, hi=hi, steps=_steps(rng, count * hi ** 3))
    n = rng.choice([16, 24, 32, 40, 48, 56, 64])
    if kind == "train":
        return dict(kind=kind, n=n, pairs=rng.choice([1, 2, 4, 8]), iters=rng.randint(5, 30))
    return dict(kind=kind, n=n, steps=rng.randint(5, 30))


# ---- inputs ------------------------------------------------------------------

def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))


def _vortex(shape, seed, mach):
    """Conserved state (5, nz + 1, ny + 1, nx + 1) on the GPU of a Taylor-Green vortex on the [0, 2 pi]-periodic box with
    8 random modes of 5% and noise of 0.1% of the Mach number per velocity component; duplicate planes agree."""
    g = _rng(seed)
    nz, ny, nx = shape
    f64 = dict(dtype=torch.float64, device="cuda")
    # gridtoy: x from 0, y from -pi, z falls from pi to -pi
    x = (2 * math.pi / nx * torch.arange(nx, **f64))[None, None, :]
    y = (2 * math.pi / ny * torch.arange(ny, **f64) - math.pi)[None, :, None]
    z = (math.pi - 2 * math.pi / nz * torch.arange(nz, **f64))[:, None, None]
    u = [mach * torch.sin(x) * torch.cos(y) * torch.cos(z), -mach * torch.cos(x) * torch.sin(y) * torch.cos(z),
         torch.zeros(nz, ny, nx, **f64)]
    for c in range(3):
        k = torch.randint(-3, 4, (8, 3), generator=g, device="cuda").tolist()
        phi = (2 * math.pi * torch.rand(8, generator=g, **f64)).tolist()
        for (kx, ky, kz), ph in zip(k, phi):
            u[c] = u[c] + 0.05 * mach / math.sqrt(8) * torch.sin(kx * x + ky * y + kz * z + ph)
        u[c] = u[c] + 1e-3 * mach * (2 * torch.rand(nz, ny, nx, generator=g, **f64) - 1)
    p = 1 / GAM + mach * mach / 16 * (torch.cos(2 * x) + torch.cos(2 * y)) * (torch.cos(2 * z) + 2)
    rho = GAM * p
    q = torch.stack([rho, rho * u[0], rho * u[1], rho * u[2],
                     p / (GAM - 1) + 0.5 * rho * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)])
    for d in (1, 2, 3):   # the last plane of each direction repeats the first
        q = torch.cat([q, q.narrow(d, 0, 1)], dim=d)
    return q


def _host(q):
    return q.reshape(q.shape[0], -1).cpu().numpy()


def _box(nx, ny, nz):
    return (nx, ny, nz, 0.0, 2 * math.pi, math.pi, 2 * math.pi)


def _instances(case, seed):
    """[(nx, ny, nz, Mach, Reynolds, seed)] of a periodic, ensemble or coarse case."""
    if case["kind"] == "periodic":
        return [(case["nx"], case["ny"], case["nz"], 0.1, 1600.0, seed)]
    if case["kind"] == "apply":
        return [(case["n"],) * 3 + (0.1, 1600.0, seed)]
    r = np.random.default_rng(seed)
    return [((case["lo"], case["hi"])[i % 3 > 0],) * 3 + (float(r.uniform(0.05, 0.3)), float(r.uniform(400, 3200)), seed + 1000 * i)
            for i in range(case["count"])]


def _periodic_case(case, seed):
    inst = _instances(case, seed)
    blocks = [dict(lxi=nx, let=ny, lze=nz, nbc=[[setup.PERIODIC] * 2] * 3, mcd=[[i, i]] * 3, inst=i)
              for i, (nx, ny, nz, *_) in enumerate(inst)]
    params = [dict(PARAMS, reoo=re / mach, viscous=int(case.get("viscous", True))) for *_, mach, re, _ in inst]
    c = Case(blocks, params, precision=CND_MIXED if case.get("mixed") else CND_FP64)
    for i, (nx, ny, nz, *_) in enumerate(inst):
        c.make_grid(i, "toy", *_box(nx, ny, nz))
    c.init_metrics()
    c.set_states([_host(_vortex((nz, ny, nx), s, mach)) for nx, ny, nz, mach, _, s in inst])
    for i in range(len(inst)):
        c.set_clock(inst=i)
    c.use_graph(case.get("graph", case["kind"] == "ensemble"))
    return c


def _pulses(c, b, g, lx, ly, lz, stream, amp, width):
    """State of block b: a uniform stream with three pressure pulses of random place; grid coordinates from the device."""
    x, y, z = torch.from_numpy(c.grid(b)).cuda()
    p = torch.full_like(x, 1 / GAM)
    for a, e, f in torch.rand(3, 3, generator=g, dtype=torch.float64, device="cuda").tolist():
        r2 = (x - x.min() - (0.2 + 0.6 * a) * lx) ** 2 + (y - y.min() - (0.2 + 0.6 * e) * ly) ** 2 + (z - z.min() - f * lz) ** 2
        p = p + amp / GAM * torch.exp(-r2 / (2 * width * width))
    rho = (GAM * p) ** (1 / GAM)
    return _host(torch.stack([rho] + [rho * v for v in stream] + [p / (GAM - 1) + 0.5 * rho * sum(v * v for v in stream)]))


def _channel_case(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    block = dict(lxi=nx, let=ny, lze=nz, mcd=[[-1, -1], [0, 0], [-1, -1]],
                 nbc=[[setup.NONREF] * 2, [setup.PERIODIC] * 2, [setup.WALL_VIS, setup.WALL_INV]])
    c = Case([block], dict(PARAMS, reoo=500.0, viscous=1))
    c.make_grid(0, "toy", nx, ny, nz, 0.0, float(nx), ny / 2.0, float(nz))
    c.init_metrics()
    c.set_states([_pulses(c, 0, _rng(seed), nx, ny, nz, (0.0, 0.2, 0.0), 1e-3, 3.0)])
    c.set_clock()
    c.record(True)
    return c


def _sheared_case(case, seed):
    nx, nx2, ny, nz = case["nx"], case["nx2"], case["ny"], case["nz"]
    pairs = [((nx, ny, nz), (nx2, ny, nz)), ((nx + nx // 3, ny // 2 + 2, nz), (nx2 - nx2 // 3, ny // 2 + 2, nz))]
    lmax = float(max(a[0] + b[0] for a, b in pairs))
    blocks = [b for p, pair in enumerate(pairs) for b in setup.sheared_pair_blocks(list(pair), first=2 * p)]
    c = Case(blocks, dict(PARAMS, reoo=1000.0, amach1=0.5, viscous=1, sponge=1, szco=0.5, szth0=0.1 * lmax,
                          szth1=0.1 * lmax, doml1=lmax))
    b = 0
    for pair in pairs:
        lx, x0 = float(pair[0][0] + pair[1][0]), 0.0
        for n in pair:
            c.make_grid(b, "sheared", x0, 1.0, 0.05, lx, float(n[1]))
            x0, b = x0 + n[0], b + 1
    c.init_metrics()
    g = _rng(seed)
    c.set_states([_pulses(c, b, g, k["lxi"], k["let"], nz, (0.5, 0.0, 0.0), 1e-3, 5.0) for b, k in enumerate(blocks)])
    c.set_clock()
    return c


def _weights(seed):
    """Flat parameters of a network in training: He-uniform weights, the last layer a tenth, small biases."""
    g, out = torch.Generator().manual_seed(int(seed) % (1 << 62)), []
    for i, (ci, co) in enumerate(zip(CHANNELS, CHANNELS[1:])):
        a = math.sqrt(6 / (27 * ci)) * (0.1 if i == 2 else 1.0)
        out += [a * (2 * torch.rand(co * 27 * ci, generator=g) - 1), 0.02 * torch.randn(co, generator=g) * (0.1 if i == 2 else 1.0)]
    return torch.cat(out).numpy()


# Normalisation of a 64^3 coarse run at Mach 0.1, as training measures it.
IN_MEAN, IN_SCALE = np.array([1.0, 0, 0, 0, 1.788]), np.array([2e-3, 0.05, 0.05, 0.05, 5e-3])
OUT_SCALE = np.array([1e-6, 1e-5, 1e-5, 1e-5, 3e-6])


def _pairs(case, seed):
    """Normalised inputs and targets (pairs, n^3, 5) in FP32."""
    g, n = _rng(seed), case["n"]
    xs, ts = [], []
    for k in range(case["pairs"]):
        q = _vortex((n, n, n), seed + 7919 * k, 0.1)[:, :n, :n, :n].reshape(5, -1).T
        x = (q - torch.from_numpy(IN_MEAN).cuda()) / torch.from_numpy(IN_SCALE).cuda()
        xs.append(x.float())
        ts.append((0.3 * x.roll(1, 0) + torch.randn(n ** 3, 5, generator=g, device="cuda")).float())
    return torch.stack(xs), torch.stack(ts)


def prepare(case, seed):
    if case["kind"] == "train":
        net = Net(case["n"], capacity=case["pairs"])
        net.set_params(_weights(seed))
        for x, t in zip(*_pairs(case, seed)):
            net.add_pair_host(x.cpu().numpy(), t.cpu().numpy())
        return dict(case=case, net=net, passes=0)
    make = {"channel": _channel_case, "sheared": _sheared_case}.get(case["kind"], _periodic_case)
    c = make(case, seed)
    c.tune()   # as the first step of any run does
    s = dict(case=case, run=c)
    if case["kind"] == "apply":
        s["net"] = Net(case["n"])
        s["net"].set_params(_weights(seed))
        s["net"].set_norm(IN_MEAN, IN_SCALE, OUT_SCALE)
    return s


def run(s):
    case = s["case"]
    if case["kind"] == "train":
        loss = s["net"].train(case["iters"], lr=1e-4, seed=s["passes"])
        s["passes"] += 1
        return dict(params=s["net"].params(), loss=loss)
    c = s["run"]
    if case["kind"] == "apply":
        for _ in range(case["steps"]):
            c.step(1)
            s["net"].apply(c, 0)
    else:
        c.step(case["steps"])
    out = dict(states=[c.state(b) for b in range(len(c.blocks))],
               clocks=np.array([list(c.clock(i).values()) for i in range(len(c.params))]))
    if case["kind"] == "channel":
        out["averages"] = c.record_read(0)
    return out


# ---- work --------------------------------------------------------------------

def work(case):
    if case["kind"] == "train":
        v = case["n"] ** 3
        l1, l2, l3 = (2 * 27 * v * a * b for a, b in zip(CHANNELS, CHANNELS[1:]))
        # forward, the data gradients of layers 3 and 2, the weight gradients; the pair is read once an iteration
        return dict(flops=case["iters"] * (2 * (l1 + l2 + l3) + l2 + l3), bytes=case["iters"] * v * (8 * 2 + 5 * 4))
    if case["kind"] == "channel":
        pts = (case["nx"] + 1) * (case["ny"] + 1) * (case["nz"] + 1)
    elif case["kind"] == "sheared":
        nx, nx2, ny, nz = case["nx"], case["nx2"], case["ny"], case["nz"]
        pts = ((nx + nx2 + 2) * (ny + 1) + (nx + nx // 3 + nx2 - nx2 // 3 + 2) * (ny // 2 + 3)) * (nz + 1)
    else:
        pts = sum((a + 1) * (b + 1) * (c + 1) for a, b, c, *_ in _instances(case, 0))
    viscous = case.get("viscous", True)
    # Bytes per point: each sweep reads its fields and writes its results once.  A step: three filter sweeps (80 each);
    # a viscous stage: the primitives (72), three gradient sweeps (64 each), fluxes from state, gradients and metrics
    # into the fluxes of two directions and the derivative along the third (336), two flux sweeps (80 and, with the
    # update, 208); an inviscid stage: fluxes from state and metrics likewise (232), two flux sweeps.
    per = 240 + 4 * ((72 + 2 * 64 + 304 if viscous else 232) + 80 + 208)
    # Operations per point: 13 of a filter right-hand side and 9 of a solve per sweep and variable; 5 and 9 of a
    # derivative; the pointwise stresses, fluxes and update.
    ops = 15 * 22 + 4 * ((27 if viscous else 15) * 14 + (250 if viscous else 100) + 25)
    w = dict(bytes=float(case["steps"] * per * pts), flops=float(case["steps"] * ops * pts))
    if case["kind"] == "apply":
        v = case["n"] ** 3
        w["flops"] += case["steps"] * sum(2.0 * 27 * v * a * b for a, b in zip(CHANNELS, CHANNELS[1:]))
        w["bytes"] += case["steps"] * 80.0 * pts
    return w


# ---- the same in 64 bits -------------------------------------------------------

def _filter_rows():
    """Interior (alpha, beta, a, b, c) and the one-sided rows (left-hand offsets -2..2, right-hand weights) of the filter."""
    kc = math.pi * FLTK
    c1, c2, c3 = (math.cos(m * kc) for m in (1, 2, 3))
    den = 30 + 5 * (7 - 8) * c1 + 2 * (1 + 4) * c2 - 3 * c3
    al, be = (-30 * c1 - 2 * c3) / den, 0.5 * (2 * (13 - 4) + (33 - 24) * c1 + 6 * c2 - c3) / den
    a = 30 * math.cos(0.5 * kc) ** 4 / den
    b, c = -2 * a / 5, a / 15
    f, lg = FLTRBC, math.log(FLTRBC)
    nrm = 1 / (1 + al * f + be * f * f)
    g0 = (f - 1) * (a + c + (f + 1) * (b + f * c)) / lg
    g1 = (f - 1) * (b + c * (f + 1)) / lg
    g2 = c * (f - 1) / lg
    left = [[0, 0, 1, al * nrm, be * nrm], [0, al + be * f, 1, al, be], [be, al, 1, al, be]]
    right = [[(a - 5 * g0 / 3) * nrm, (b + 10 * g0 / 21) * nrm, (c - 5 * g0 / 42) * nrm, 5 * g0 / 252 * nrm, -g0 / 630 * nrm],
             [a + b + c + 1627 * g1 / 1260, a + 10 * g1 / 21, b - 5 * g1 / 42, c + 5 * g1 / 252, -g1 / 630],
             [b + c + 1627 * g2 / 1260, a - 5 * g2 / 3, a - 5 * g2 / 42, b + 5 * g2 / 252, c - g2 / 630]]
    return (al, be, a, b, c), left, right


def _line_operators(n):
    """Dense (n + 1, n + 1) derivative and filter of a line of n cells that is its own periodic partner: the interior
    rows, and at both ends the closure that two half-lines of 12 points, solved together with one-sided outer rows,
    give when the couplings across their interface move to the right-hand side."""
    A0 = (-6.666666667794732, 9.000000000052879, 1.333333333178555, -0.0833333333455545)
    A1 = (-0.3506944444280639, 0.8249999999974599, 0.7444444444773477, 0.014583333334139971)
    (al, be, fa, fb, fc), left, right = _filter_rows()
    found = []
    for filt in (False, True):
        a1, a2 = (al, be) if filt else (4 / 9, 1 / 36)
        rhs = [fc, fb, fa, -2 * (fa + fb + fc), fa, fb, fc] if filt else [0, -25 / 216, -20 / 27, 0, 20 / 27, 25 / 216, 0]
        A, B = np.zeros((24, 24)), np.zeros((24, 24))
        for i in range(3, 21):
            A[i, i - 2:i + 3], B[i, i - 3:i + 4] = [a2, a1, 1, a1, a2], rhs
        sign = 1 if filt else -1
        if filt:
            for r in range(3):
                A[r, :r + 3] = left[r][2 - r:]
                B[r, [c for c in range(6) if c != r]] = right[r]
                B[r, r] = -sum(right[r])
        else:
            A[0, :3], B[0, :5] = [1, 8.000000000449464, 6.000000000542], [-sum(A0), *A0]
            A[1, :4], B[1, :5] = [0.09166666665902128, 1, 1.3500000000438646, 0.2666666666794667], [A1[0], -sum(A1), *A1[1:]]
            A[2, :5], B[2, :5] = [a2, a1, 1, a1, a2], rhs[1:6]
        for r in range(3):
            A[23 - r], B[23 - r] = A[r, ::-1], sign * B[r, ::-1]
        R = A.copy()
        R[10, 12] = R[11, 12] = R[11, 13] = R[13, 11] = R[12, 11] = R[12, 10] = 0
        M = (R @ np.linalg.solve(A, B))[12:14]
        own, other = M[:, 12:], M[:, 11::-1]      # by the distance from the interface
        L, W = np.zeros((n + 1, n + 1)), np.zeros((n + 1, n + 1))
        for i in range(n + 1):
            for o, v in zip(range(-2, 3), (a2, a1, 1, a1, a2)):
                if 0 <= i + o <= n:
                    L[i, i + o] = v
            for o, v in zip(range(-3, 4), rhs):
                W[i, (i + o) % n if i + o < 0 or i + o > n else i + o] += v
        for r in range(2):                        # the partner's points start one behind its own end
            row = np.zeros(n + 1)
            np.add.at(row, np.arange(12), own[r])
            np.add.at(row, n - 1 - np.arange(12), other[r])
            W[r], W[n - r] = row, sign * row[::-1]
        X = np.linalg.solve(L, W)
        found.append(torch.from_numpy(X + np.eye(n + 1) if filt else X).cuda())
    return found


def _along(M, f, d):
    """M applied along direction d (0: x, the last axis) of fields (..., nz, ny, nx)."""
    if d == 0:
        return f @ M.T
    if d == 1:
        return M @ f
    return (M @ f.flatten(-2)).unflatten(-1, f.shape[-2:])


class _Flow:
    """One periodic block of the exact time loop."""

    def __init__(self, nx, ny, nz, mach, re, seed, viscous):
        self.q = _vortex((nz, ny, nx), seed, mach)
        lines = {n: _line_operators(n) for n in {nx, ny, nz}}
        self.fd, self.fi = ([lines[n][k] for n in (nx, ny, nz)] for k in (0, 1))
        self.h = [nx / (2 * math.pi), ny / (2 * math.pi), -nz / (2 * math.pi)]   # d(index)/d(coordinate)
        self.viscous = viscous
        self.s0 = 111 / TEMPOO
        self.mu0 = (self.s0 + 1) / (re / mach)
        self.n = self.ndt = 0
        self.dt = self.dts = self.dte = self.time = 0.0

    def primitives(self, q):
        u = [q[c] / q[0] for c in (1, 2, 3)]
        p = (GAM - 1) * (q[4] - 0.5 * sum(q[c + 1] * u[c] for c in range(3)))
        T = GAM * p / q[0]
        return u, p, T, self.mu0 * T ** 1.5 / (T + self.s0)

    def schedule(self):
        if self.n % 10 == 1:
            u, _, T, mu = self.primitives(self.q)
            hh = sum(h * h for h in self.h)
            speed = torch.sqrt(T * hh) + sum((v * h).abs() for v, h in zip(u, self.h))
            self.ndt, self.dts = self.n, self.dte
            self.dte = CFL / float(speed.max())
            if self.viscous:
                self.dte = min(self.dte, 0.5 / float((mu * hh / self.q[0]).max()))
        self.dt = self.dts + (self.dte - self.dts) * math.sin(0.05 * math.pi * (self.n - self.ndt)) ** 2

    def rate(self, q):
        """Sum of the flux derivatives in coordinates."""
        u, p, T, mu = self.primitives(q)
        tau = None
        if self.viscous:
            v = torch.stack(u + [T])
            g = [h * _along(M, v, d) for d, (M, h) in enumerate(zip(self.fd, self.h))]      # g[d][component]
            div = g[0][0] + g[1][1] + g[2][2]
            tau = [[mu * (g[d][c] + g[c][d] - (2 / 3 * div if c == d else 0)) for c in range(3)] for d in range(3)]
            heat = [mu / ((GAM - 1) * PRANDTL) * g[d][3] for d in range(3)]
            del v, g, div
        out = torch.zeros_like(q)
        for d in range(3):
            f = torch.stack([q[c] * u[d] for c in range(4)] + [(q[4] + p) * u[d]])
            f[d + 1] += p
            if tau:
                for c in range(3):
                    f[c + 1] -= tau[d][c]
                    f[4] -= tau[d][c] * u[c]
                f[4] -= heat[d]
            out += self.h[d] * _along(self.fd[d], f, d)
        return out

    def step(self):
        for d in (1, 2, 0):
            self.q = _along(self.fi[d], self.q, d)
        self.schedule()
        start = self.q
        for nk in range(1, 5):
            self.q = start - self.dt / (5 - nk) * self.rate(self.q)
            # a point on periodic faces becomes the mean of itself and its copy across each of them
            total, count = self.q.clone(), torch.ones_like(self.q[:1])
            for d in (1, 2, 3):
                for end in (0, -1):
                    total.select(d, end).add_(self.q.select(d, -1 - end))
                    count.select(d, end).add_(1)
            self.q = total / count
        self.n += 1
        self.time += self.dt

    def clock(self):
        return [self.n, self.ndt, self.dt, self.dts, self.dte, self.time]


def _net64(x, w, n):
    """The network on (n^3, 5) normalised inputs with flat parameters w, in w's precision."""
    a, at = x, 0
    for i, (ci, co) in enumerate(zip(CHANNELS, CHANNELS[1:])):
        W = w[at:at + co * 27 * ci].reshape(co, 27, ci)
        b = w[at + co * 27 * ci:at + co * 27 * ci + co]
        at += co * 27 * ci + co
        grid, y = a.reshape(n, n, n, ci), b
        for t in range(27):
            dx, dy, dz = t % 3 - 1, t // 3 % 3 - 1, t // 9 - 1
            y = y + grid.roll((-dz, -dy, -dx), (0, 1, 2)).reshape(-1, ci) @ W[:, t].T
        a = torch.relu(y) if i < 2 else y
    return a


class _Mt64:
    """The 64-bit Mersenne Twister of the C++ standard library, which draws the training pairs."""

    def __init__(self, seed):
        m = (1 << 64) - 1
        self.s = [seed & m]
        for i in range(1, 312):
            self.s.append((6364136223846793005 * (self.s[-1] ^ (self.s[-1] >> 62)) + i) & m)
        self.i = 312

    def next(self):
        if self.i == 312:
            s = self.s
            for k in range(312):
                x = (s[k] & 0xFFFFFFFF80000000) | (s[(k + 1) % 312] & 0x7FFFFFFF)
                s[k] = s[(k + 156) % 312] ^ (x >> 1) ^ (0xB5026F5AA96619E9 if x & 1 else 0)
            self.i = 0
        x = self.s[self.i]
        self.i += 1
        x ^= (x >> 29) & 0x5555555555555555
        x ^= (x << 17) & 0x71D67FFFEDA60000
        x ^= (x << 37) & 0xFFF7EEE000000000
        return x ^ (x >> 43)


def exact(case, seed):
    if case["kind"] in ("channel", "sheared"):
        return None   # characteristic faces and sponge have no short restatement
    if case["kind"] == "train":
        x, t = (v.double() for v in _pairs(case, seed))
        w = torch.from_numpy(_weights(seed)).double().cuda().requires_grad_()
        m1, m2, total, pick = torch.zeros_like(w), torch.zeros_like(w), 0.0, _Mt64(0)
        for it in range(1, case["iters"] + 1):
            k = pick.next() * case["pairs"] >> 64   # a power of two of pairs: the top bits
            loss = ((_net64(x[k], w, case["n"]) - t[k]) ** 2).mean()
            g, = torch.autograd.grad(loss, w)
            total += float(loss)
            m1, m2 = 0.9 * m1 + 0.1 * g, 0.999 * m2 + 0.001 * g * g
            with torch.no_grad():
                w -= 1e-4 * (m1 / (1 - 0.9 ** it)) / ((m2 / (1 - 0.999 ** it)).sqrt() + 1e-8)
        return dict(params=w.detach().cpu().numpy(), loss=total / case["iters"])
    flows = [_Flow(*inst, case.get("viscous", True)) for inst in _instances(case, seed)]
    if case["kind"] == "apply":
        n, w = case["n"], torch.from_numpy(_weights(seed)).double().cuda()
        mean, scale, out = (torch.from_numpy(v).cuda() for v in (IN_MEAN, IN_SCALE, OUT_SCALE))
    for f in flows:
        for _ in range(case["steps"]):
            f.step()
            if case["kind"] == "apply":
                y = _net64((f.q[:, :n, :n, :n].reshape(5, -1).T - mean) / scale, w, n) * out
                y = y.T.reshape(5, n, n, n)
                for d in (1, 2, 3):
                    y = torch.cat([y, y.narrow(d, 0, 1)], dim=d)
                f.q = f.q + y
    return dict(states=[_host(f.q) for f in flows], clocks=np.array([f.clock() for f in flows]))
