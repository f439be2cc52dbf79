"""Reciprocal and square root of the FP64 fast forms, on the CPU.

The GPU gives estimates (v_rcp_f64, v_rsq_f64); engine.hpp refines them.  The refinement is plain C++ and
is run here from estimates off by up to 2^-23, against long double: within one unit of 2^-53 of the value
(half a unit in the last place at the low end of a binade), plus 2^-60 for what the steps leave.
"""
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "dgswemv2_amd" / "csrc"

PROGRAM = r"""
#include <math.h>
#include <cmath>
#include <cstdio>
#include <random>

#include "engine.hpp"
int main() {
    std::mt19937_64 rng(7);
    std::uniform_real_distribution<double> mant(1.0, 4.0), off(-1.0, 1.0);
    long double worst_r = 0, worst_s = 0;
    for (int i = 0; i < 2000000; ++i) {
        const double x = std::ldexp(i % 97 ? mant(rng) : 1.0 + 0x1p-52 * (i % 1000), 2 * (i % 41 - 20));
        const double d = (i % 3 ? off(rng) : (i % 2 ? 1.0 : -1.0)) * 0x1p-23;
        const long double r = 1.0L / x, s = std::sqrt((long double)x);
        worst_r = std::fmax(worst_r, std::fabs(rkdg::rcp_refined(x, (double)(r * (1 + d))) / r - 1));
        worst_s = std::fmax(worst_s, std::fabs(rkdg::root_refined(x, (double)((1 + d) / s)) / s - 1));
    }
    std::printf("%.4f %.4f\n", (double)(worst_r * 0x1p53L), (double)(worst_s * 0x1p53L));
}
"""


def test_refined_reciprocal_and_root(tmp_path):
    subprocess.run(["make", "-C", str(CSRC), "_build/device_tables.h"], check=True, capture_output=True)
    src, exe = tmp_path / "roots.cpp", tmp_path / "roots"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-w", f"-I{CSRC}", f"-I{CSRC / '_build'}", str(src), "-o", str(exe)],
                   check=True)
    r, s = (float(z) for z in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split())
    print("units of 2^-53: reciprocal", r, "root", s)
    assert r <= 1.0 + 2.0**-7 and s <= 1.0 + 2.0**-7
