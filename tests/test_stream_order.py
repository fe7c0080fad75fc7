"""Order of a context's first work after its creation, on the CPU with a HIP
runtime that only keeps the order (hip_order_stub.cpp): nothing a context runs
on its own stream may meet a clear on the null stream that nothing has waited
for.  Blocks with and without entries of the junction averaging, whose upload
waits by itself."""
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
mcd, nbc = {mcd}, {nbc}
n = len(mcd)
c = Case([dict(lxi=14, let=13, lze=12, nbc=nbc[b], mcd=mcd[b]) for b in range(n)], dict(reoo=100.0))
for b in range(n):
    c.make_grid(b, "toy", 14, 13, 12, 0.0, 1.0, 1.0, 1.0)
c.init_metrics()
c.step(2)
stub = ctypes.CDLL({stub!r})
print("launches", stub.order_launches(), "violations", stub.order_violations())
"""

SELF = ([[[0, 0]] * 3], [[[45, 45]] * 3])                                   # its own partner: no junction entries
FREE = ([[[-1, -1]] * 3], [[[10, 10]] * 3])                                 # no averaged face
PAIR = ([[[1 - b, 1 - b], [b, b], [b, b]] for b in range(2)], [[[45, 45]] * 3] * 2)


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "hip_order_stub.cpp"), "-o", so], check=True)
    return so


@pytest.mark.parametrize("case", [SELF, FREE, PAIR], ids=["self", "free", "pair"])
def test_first_work_of_a_context_is_ordered(stub, case):
    code = CHILD.format(root=ROOT, stub=stub, mcd=case[0], nbc=case[1])
    preload = " ".join([stub] + os.environ.get("LD_PRELOAD", "").split())   # in front of what is there
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, LD_PRELOAD=preload, CANARD_TUNE="0"),
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    word = r.stdout.split()
    assert int(word[1]) > 20, r.stdout    # the stub took the calls
    assert int(word[3]) == 0, r.stdout
