"""Where blending leaves entries out, on the host: the functions of blend_cuts.hpp compiled with g++
(no contraction, as the library) against what they stand for, evaluated directly."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "threedgaussiansplatting.jl_amd", "csrc")


def run_cpp(tmp_path, source):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text('#include <cstdio>\n#include <random>\n#include "blend_cuts.hpp"\nusing namespace tdgs;\n' + source)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()


@pytest.mark.parametrize("length", [1, 30, 100, 300, 1000, 3000, 100000])
def test_nothing_outside_the_box_reaches_the_cut(length, tmp_path):
    """Backward blending's boxes against its walk of every entry: no pixel outside a Gaussian's box has an
    exponent, as the walk computes it in float, that reaches the cut; from round Gaussians to needles, around the
    points where the box touches the ellipse (the walk's rounding reaches farthest there) and anywhere."""
    out = run_cpp(tmp_path, """
int main() {
    std::mt19937 rng(1);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    std::normal_distribution<double> N(0.0, 1.0);
    const double L = %d;
    long bad = 0, outside = 0;
    for (int i = 0; i < 100000; ++i) {
        const double th = 3.141592653589793 * U(rng), s1 = L * (0.5 + 0.5 * U(rng)), s2 = U(rng), c = cos(th), s = sin(th);
        const double a = c * c * s1 * s1 + s * s * s2 * s2 + 0.3, b = c * s * (s1 * s1 - s2 * s2),
                     d = s * s * s1 * s1 + c * c * s2 * s2 + 0.3, det = a * d - b * b;
        const float A = -0.5f * kLog2e * (float)(d / det), B = -kLog2e * (float)(-b / det), C = -0.5f * kLog2e * (float)(a / det);
        const float cut = kLog2e * ((float)(log(1.0 / 255.0) - 1e-3) - log_f((float)(0.05 + 0.95 * U(rng))));
        float rx, ry;
        cut_box(A, B, C, cut, &rx, &ry);
        if (!(rx < kInf) || !(ry < kInf)) continue;
        for (int k = 0; k < 12; ++k) {
            const float sign = U(rng) < 0.5 ? -1.0f : 1.0f, f = (float)(1.0 + 0.02 * U(rng) * U(rng)), e = (float)(0.7 * N(rng));
            float du, dv;   // past the box on the left or right, on top or below, or both
            if (k < 5) { du = sign * rx * f; dv = (float)(-(double)B / (2.0 * C) * du + e); }
            else if (k < 10) { dv = sign * ry * f; du = (float)(-(double)B / (2.0 * A) * dv + e); }
            else { du = sign * rx * f; dv = (float)(2.0 * (U(rng) - 0.5)) * ry; }
            if (!(fabsf(du) > rx) && !(fabsf(dv) > ry)) continue;
            ++outside;
            const float x = fmaf(fmaf(A, du, B * dv), du, C * dv * dv);
            if (!(x < cut)) ++bad;
        }
    }
    printf("%%ld %%ld\\n", bad, outside);
}
""" % length)
    bad, outside = map(int, out)
    assert bad == 0 and (outside > 100_000 or length == 100000), (bad, outside)
