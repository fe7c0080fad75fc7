"""A launch of eta and zeta sweeps together is only made where its LDS fits
(joint_lds_check.cpp, host code only)."""
import os
import subprocess

from canard_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_joint_launch_fits_the_lds(tmp_path):
    exe = str(tmp_path / "joint_lds")
    subprocess.run([build.hipcc(), "-O1", "-std=c++17", "-x", "hip", "--offload-host-only",
                    os.path.join(HERE, "joint_lds_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
