"""Junction entries that average a point with copies of itself only are
dropped (drop_self_averages, canard_amd/csrc/cnd_scheme.cpp): none is left on
a block that is its own periodic partner, all are left where blocks meet
others, and every dropped entry's average equals the point to the rounding of
its sum (at most 8 terms: 8 ulp).  Host logic only: compiled with g++ and run
on the CPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(os.path.dirname(HERE), "canard_amd", "csrc")

PROGRAM = r"""
#include <cmath>
#include "junction_program_check.cpp"
int drop(const char *name, const std::vector<BlockSpec> &blocks, bool all, bool none)
{
    std::vector<int64_t> off;
    int64_t NT = 0;
    for (const BlockSpec &b : blocks) { off.push_back(NT); NT += int64_t(b.n[0]) * b.n[1] * b.n[2]; }
    JunctionPlan pc, pe;
    junction_plans(blocks, off, pc, pe);
    JunctionProgram J = junction_program(pc, pe), D = J;
    const int left = drop_self_averages(D);
    int before = 0, bad = 0;
    for (int w : J.write) before += w;
    std::mt19937_64 rng(3);
    std::uniform_real_distribution<double> u(0.5, 1.5);
    std::vector<double> q(5 * size_t(NT));
    for (double &x : q) x = u(rng);
    std::vector<double> a = q, b = q;
    apply_program(J, a, NT);
    apply_program(D, b, NT);
    for (size_t i = 0; i < q.size(); ++i) bad += !(std::abs(a[i] - b[i]) <= 8 * 2.3e-16 * std::abs(a[i]));
    std::printf("%s before %d left %d bad %d\n", name, before, left, bad);
    return bad || (all && left) || (none && left != before) || before == 0;
}
int junction_drop_main()
{
    int fails = 0;
    BlockSpec p = blk(13, 14, 15, 45, 45, 45), q = p;
    for (int d = 0; d < 3; ++d) { p.partner[d][0] = p.partner[d][1] = 0; q.partner[d][0] = q.partner[d][1] = 1; }
    fails += drop("one", {p}, true, false);
    fails += drop("two_instances", {p, q}, true, false);
    std::vector<BlockSpec> v;
    auto id = [](int i, int j, int k) { return i + 2 * j + 4 * k; };
    for (int k = 0; k < 2; ++k)
        for (int j = 0; j < 2; ++j)
            for (int i = 0; i < 2; ++i) {
                BlockSpec b = blk(13, 14, 15, 35, 35, 35);
                b.partner[0][0] = b.partner[0][1] = id(1 - i, j, k);
                b.partner[1][0] = b.partner[1][1] = id(i, 1 - j, k);
                b.partner[2][0] = b.partner[2][1] = id(i, j, 1 - k);
                v.push_back(b);
            }
    fails += drop("eight", v, false, true);
    return fails;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_self_averages_are_dropped(tmp_path):
    src = tmp_path / "drop.cpp"
    src.write_text("#define main junction_program_main\n" + PROGRAM + "#undef main\nint main() { return junction_drop_main(); }\n")
    exe = tmp_path / "drop"
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-I", SRC, "-I", HERE, str(src),
                    os.path.join(SRC, "cnd_scheme.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
