"""Reads of a state into page-locked memory: every byte at the sizes of the
chunked reads, at the start and inside of the caller's allocation, and by a
plain copy.  The chunked read allocates 48 MiB of staging memory with a
context's first one, so the plain copy shows in the process's address space,
which then grows by less than that; a read into pageable memory shows that the
measurement sees it."""
import ctypes as C

import numpy as np
import pytest

from canard_amd import cases
from canard_amd.solver import Case

pytestmark = pytest.mark.gpu

MIB = 1 << 20


class PageLocked:
    """n doubles from hipHostMalloc of the HIP runtime the library uses."""

    def __init__(self, n):
        self.hip, self.p = C.CDLL("libamdhip64.so.7"), C.c_void_p()
        self.hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
        self.hip.hipHostFree.argtypes = [C.c_void_p]
        assert self.hip.hipHostMalloc(C.byref(self.p), 8 * n, 0) == 0
        self.a = np.ctypeslib.as_array(C.cast(self.p, C.POINTER(C.c_double)), (n,))
        self.a[:] = 0.0

    def free(self):
        assert self.hip.hipHostFree(self.p) == 0


def _address_space():
    with open("/proc/self/statm") as f:
        return int(f.read().split()[0]) * 4096


def _case(nxyz, seed):
    lx, ly, lz = nxyz
    c = Case([cases.periodic_block(0, lxi=lx, let=ly, lze=lz)], dict(reoo=1600.0))
    q = np.random.default_rng(seed).random((5, (lx + 1) * (ly + 1) * (lz + 1)))
    c.set_states([q])
    return c, q


def _read(c, dst):
    assert c.L.cnd_get_state(c.h, 0, dst.ctypes.data_as(C.POINTER(C.c_double))) == 0


@pytest.mark.parametrize("nxyz", [(12, 12, 12), (93, 93, 93), (94, 94, 94), (127, 127, 127), (150, 129, 60)])
@pytest.mark.parametrize("offset", [0, 1, 513])
def test_reads_into_page_locked_memory(nxyz, offset):
    c, q = _case(nxyz, 3)
    print(f"[read] {nxyz} page-locked, offset {offset}", flush=True)
    locked = PageLocked(q.size + offset + 7)
    mem = locked.a
    dst = mem[offset:offset + q.size]
    for _ in range(2):
        _read(c, dst)
        assert np.array_equal(dst.reshape(q.shape), q)
        assert not mem[:offset].any() and not mem[offset + q.size:].any()
        dst[:] = 0.0
    c.close()
    locked.free()


def test_page_locked_memory_takes_a_plain_copy():
    nxyz = (110, 110, 110)
    first, q = _case(nxyz, 4)   # what the runtime allocates with the first copies of a process
    locked = PageLocked(5 * 111 ** 3)
    mem, pageable = locked.a.reshape(5, 111 ** 3), np.zeros((5, 111 ** 3))
    _read(first, mem)
    _read(first, pageable)
    first.close()
    grown = {}
    for name, dst in (("page-locked", mem), ("pageable", pageable)):
        c, q = _case(nxyz, 5)
        before = _address_space()
        _read(c, dst)
        grown[name] = _address_space() - before
        assert np.array_equal(dst, q)
        c.close()
    locked.free()
    print("[read] address space grown by", grown, flush=True)
    assert grown["pageable"] >= 40 * MIB, grown
    assert grown["page-locked"] < 16 * MIB, grown
