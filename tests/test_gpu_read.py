"""Reads of a state in the caller's memory, below and above the size from
which they go through pinned chunks: every byte of what was set, at chunk
remainders of every kind, into an unaligned destination, after queued work,
and from two contexts at once."""
import ctypes as C
import threading

import numpy as np
import pytest

from canard_amd import cases
from canard_amd.solver import Case

pytestmark = pytest.mark.gpu


def _case(nxyz, seed):
    lx, ly, lz = nxyz
    c = Case([cases.periodic_block(0, lxi=lx, let=ly, lze=lz)], dict(reoo=1600.0))
    q = np.random.default_rng(seed).random((5, (lx + 1) * (ly + 1) * (lz + 1)))
    c.set_states([q])
    return c, q


# 94^3, 95^3: either side of 32 MiB; 128^3: whole chunks of 16 MiB per
# variable; 129^3, 257 x 130 x 61: remainders
@pytest.mark.parametrize("nxyz", [(12, 12, 12), (93, 93, 93), (94, 94, 94), (127, 127, 127), (128, 128, 128),
                                  (256, 129, 60)])
def test_state_reads_every_byte(nxyz):
    c, q = _case(nxyz, 1)
    print(f"[read] {nxyz}", flush=True)
    for _ in range(2):
        assert np.array_equal(c.state(0), q)
    raw = np.zeros(q.nbytes + 24, dtype=np.uint8)   # destination at an odd multiple of 8 bytes, with guards
    dst = raw[8:8 + q.nbytes].view(np.float64)
    assert c.L.cnd_get_state(c.h, 0, dst.ctypes.data_as(C.POINTER(C.c_double))) == 0
    assert np.array_equal(dst.reshape(q.shape), q)
    assert not raw[:8].any() and not raw[-16:].any()
    c.close()


def test_reads_of_two_contexts_and_after_queued_steps():
    made = [_case((100, 96, 99), s) for s in (1, 2)]
    got = [None, None]

    def read(i):
        for _ in range(3):
            got[i] = made[i][0].state(0)

    threads = [threading.Thread(target=read, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(2):
        assert np.array_equal(got[i], made[i][1])
        made[i][0].close()
    lx, ly, lz = 100, 96, 99
    xyz = cases.gridtoy(lx, ly, lz, doml0=0.0, doml1=2 * np.pi, domh=np.pi, span=2 * np.pi)
    c = Case([cases.periodic_block(0, lxi=lx, let=ly, lze=lz)], dict(reoo=1.6e4))
    c.set_grids([xyz])
    c.set_states([cases.tgv_state(xyz, (lx + 1, ly + 1, lz + 1), mach=0.1, pert=1e-3)])
    c.set_clock()
    c.step(5)
    a = c.state(0)
    assert np.array_equal(a, c.state(0)) and np.all(np.isfinite(a))
    c.close()
