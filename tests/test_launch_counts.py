"""The section timers' launch counts, on the CPU with a HIP runtime without a
device (hip_order_stub.cpp) that counts every launch: the sections of a step
hold all of its kernels but the bookkeeping of accelerating frames and of
steps that no averaging ends.  Blocks that share every launch, blocks of
unlike length, which split the segmented sweeps into one launch per class
(512 workgroups or more each), tiled directions, junctions between blocks,
walls and inviscid stages."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

CHILD = """
import ctypes, sys
sys.path.insert(0, {root!r})
from canard_amd.solver import Case
sizes, mcd, nbc, params, shapes = {case!r}
c = Case([dict(lxi=x, let=y, lze=z, nbc=nbc[b], mcd=mcd[b]) for b, (x, y, z) in enumerate(sizes)],
         dict(dict(reoo=100.0), **params))
for b, s in enumerate(sizes):
    c.make_grid(b, "toy", *s, 0.0, 1.0, 1.0, 1.0)
c.init_metrics()
for kind, d, sh in shapes:
    c.set_shape(kind, d, sh)
stub = ctypes.CDLL({stub!r})
c.profile(True)
before = stub.order_launches()
c.step(3)
print("launches", stub.order_launches() - before, "sections", *[n for _, n in c.profile_read().values()])
"""

PER = [[45, 45]] * 3


def _own(n):
    return [[[b, b]] * 3 for b in range(n)], [PER] * n


XI4 = [(k, 0, 19) for k in ("filter", "flux")]   # 4 pencils a workgroup: many tiles
CASES = {
    "one block": ([(14, 13, 12)], *_own(1), {}, []),
    "inviscid": ([(14, 13, 12)], *_own(1), dict(viscous=0), []),
    "unlike lengths": ([(150, 46, 46), (40, 46, 46)], *_own(2), {}, XI4),
    "unlike lengths, inviscid": ([(150, 46, 46), (40, 46, 46)], *_own(2), dict(viscous=0), XI4),
    "tiled": ([(14, 13, 12)], *_own(1), {}, [(k, d, -1) for k in ("filter", "grad", "flux") for d in range(3)]),
    "tiled inviscid": ([(14, 13, 12)], *_own(1), dict(viscous=0), [("flux", d, -1) for d in range(3)]),
    "two blocks": ([(14, 13, 12)] * 2, [[[1 - b, 1 - b], [b, b], [b, b]] for b in range(2)], [PER] * 2, {}, []),
    "walls": ([(14, 13, 12)], [[[-1, -1], [0, 0], [-1, -1]]], [[[10, 25], [45, 45], [20, 25]]], {}, []),
    "frame": ([(14, 13, 12)], *_own(1), dict(nsmf=0, timf=1.0, amach1=0.1), []),
}
# outside the sections, a step: k_end_step where no self-averaging kernel ends
# it, and the frame velocity of each stage
OUTSIDE = {"two blocks": 1, "frame": 5}


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "hip_order_stub.cpp"), "-o", so], check=True)
    return so


@pytest.mark.parametrize("name", CASES)
def test_sections_count_every_launch(stub, name):
    code = CHILD.format(root=ROOT, stub=stub, case=CASES[name])
    preload = " ".join([stub] + os.environ.get("LD_PRELOAD", "").split())   # in front of what is there
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, LD_PRELOAD=preload, CANARD_TUNE="0"),
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    word = r.stdout.split()
    total, sections = int(word[1]), [int(v) for v in word[3:]]
    print(name, total, sections)
    assert total == sum(sections) + 3 * OUTSIDE.get(name, 0), (total, sections)
    if name.startswith("unlike"):   # eta and zeta filters one launch each, xi one per class
        assert sections[0] == 3 * 4
