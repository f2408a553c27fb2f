"""md-bench_amd/csrc/fp64.h on the CPU: the same operations from estimates that are off by up to 5e-8,
as the hardware's may be."""
import os
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP_H = """
#pragma once
#include <cmath>
#define __device__
extern double g_off;  // relative error of the estimates
#define __builtin_amdgcn_rcp(d) (1.0 / (d) * (1.0 + g_off))
#define __builtin_amdgcn_rsq(d) (1.0 / std::sqrt(d) * (1.0 + g_off))
using std::fma;
using std::fmax;
"""

MAIN = """
#include <cstdio>
#include "fp64.h"
double g_off = 0.0;
int main()
{
    double r, worst = 0.0, rdiff = 0.0;
    long wrong = 0;
    // the arguments nearest to powers of two, but for the mantissa of all ones
    for (g_off = -5e-8; g_off <= 5e-8; g_off += 1e-9)
        for (int e = -4; e <= 4; e++)
            for (int m = 2; m <= 512; m++)
                for (int up = 0; up < 2; up++) {
                    const double d = std::ldexp(1.0 + (up ? 2 : -1) * m * 0x1p-53, e);
                    wrong += mdg::recip_rounded(d) != 1.0 / d;
                    worst = std::fmax(worst, std::fabs(mdg::recip_normal(d) * d - 1.0));
                    const double h = mdg::root_recip_normal(d, &r);
                    rdiff = std::fmax(rdiff, std::fabs(r / std::sqrt(d) - 1.0));
                    worst = std::fmax(worst, std::fabs(h * std::sqrt(d) - 1.0));
                }
    g_off = 0.0;
    const double h0 = mdg::root_recip_normal(0.0, &r);
    std::printf("%ld %g %g %g %d\\n", wrong, worst, rdiff, r, std::isfinite(h0));
}
"""


def test_reciprocals_and_roots(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP_H)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", str(tmp_path), "-I",
                    os.path.join(REPO, "md-bench_amd", "csrc"), str(tmp_path / "main.cpp"), "-o", exe],
                   check=True, timeout=120)
    out = subprocess.run([exe], check=True, timeout=120, capture_output=True, text=True).stdout.split()
    wrong, worst, rdiff, r0, finite0 = int(out[0]), *map(float, out[1:4]), int(out[4])
    assert wrong == 0
    assert worst <= 3 * 2.0 ** -53 and rdiff <= 2.0 ** -52  # an ulp, and the check's own rounding
    # a pair at distance zero: its root picks a table row, its reciprocal is no number
    assert r0 == 0.0 and not finite0
