"""The closure's kernels on every tile shape they choose by grid size: wave
rows of 8, 16 and 32 voxels (n = 24 and 56; 16 and 80; 32 and 64), tiles of
one and two planes per wave (from 56 on), one and several tiles per
workgroup, against the same network in FP64 (torch) with the activations and
weights rounded to BF16 where the device stores them.

Tolerances of the field's max norm: forward 2e-3 as in test_gpu_closure
(FP32 accumulation and rounding flips of single BF16 values).  Gradients
1e-2: the reference leaves the back-propagated gradients unrounded, the
device rounds them to BF16 (2^-9 each, averaged over the sums).  Single
input gradients are not compared: a rounding flip of one activation may
decide a ReLU the other way and change those next to it by its whole share.
Loss: 1e-3."""
import numpy as np
import pytest

import closure_ref as R

pytestmark = pytest.mark.gpu


def _round(torch, a):
    return a + (a.to(torch.bfloat16).double() - a).detach()


def _forward(torch, w, x, n):
    a, at = _round(torch, x), 0
    for i, (ci, co) in enumerate(((5, 32), (32, 32), (32, 5))):
        W = _round(torch, w[at:at + co * 27 * ci]).reshape(co, 27, ci)
        y = w[at + co * 27 * ci:at + co * 27 * ci + co]
        at += co * 27 * ci + co
        g = a.reshape(n, n, n, ci)
        for t in range(27):
            y = y + g.roll((1 - t // 9, 1 - t // 3 % 3, 1 - t % 3), (0, 1, 2)).reshape(-1, ci) @ W[:, t].T
        a = _round(torch, torch.relu(y)) if i < 2 else y
    return a


@pytest.mark.parametrize("n", [16, 24, 32, 56, 64, 80])
def test_network_matches_fp64(n):
    import torch
    from canard_amd.closure import Net
    print(f"[closure sizes] n={n}", flush=True)
    rng = np.random.default_rng(n)
    p = R.init_params(rng, gain3=1.0).astype(np.float32)
    x = rng.standard_normal((n ** 3, 5)).astype(np.float32)
    gy = rng.standard_normal((n ** 3, 5)).astype(np.float32)
    net = Net(n, capacity=1)
    net.set_params(p)
    w = torch.from_numpy(p).double().requires_grad_()
    xt = torch.from_numpy(x).double()
    yr = _forward(torch, w, xt, n)
    gyt = torch.from_numpy(gy).to(torch.bfloat16).double()
    gpr = torch.autograd.grad((yr * gyt).sum(), w)[0].numpy()
    yr = yr.detach().numpy()
    e = np.max(np.abs(net.forward(x) - yr)) / np.max(np.abs(yr))
    assert e < 2e-3, e
    gp = net.grad(x, gy)[1]
    for i in range(6):
        a, b = R.OFFS[i], R.OFFS[i + 1]
        assert np.max(np.abs(gp[a:b] - gpr[a:b])) < 1e-2 * np.max(np.abs(gpr[a:b])), i
    net.add_pair_host(x, gy)
    want = float(np.mean((yr - gy) ** 2))
    assert abs(net.eval() - want) < 1e-3 * want
    net.close()
