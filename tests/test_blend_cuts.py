"""Where blending leaves entries out, on the host: the functions of blend_cuts.hpp compiled with g++
(no contraction, as the library) against what they stand for, evaluated directly."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "threedgaussiansplatting.jl_amd", "csrc")


def run_cpp(tmp_path, source):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text('#include <cstdio>\n#include <random>\n#include <vector>\n#include "blend_cuts.hpp"\nusing namespace tdgs;\n' + source)
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


def test_exact_exponent_cut_separates_the_alphas(tmp_path):
    """The forward pass asks e >= cut instead of exp_f(e) >= min_alpha: the two agree for every one of 800 neighbouring
    exponents around the cut, for thresholds over the whole range, and next to the powers of e, 1/255, 1/2, the range's
    ends and the thresholds whose exponents change binade. A threshold may have no such cut (the kernel then compares
    alphas), but hardly any has none."""
    out = run_cpp(tmp_path, """
long bad = 0, none = 0, all = 0;
void look(float m) {
    if (!(m > 1.9e-35f) || !(m <= 0.9f)) return;
    float cut;
    ++all;
    if (!exact_exponent_cut(m, 0.99f, &cut)) { ++none; return; }
    for (int k = -400; k <= 400; ++k) {
        const float e = bits_float(float_bits(cut) - (uint32_t)k);   // (negative: k floats up)
        if ((exp_f(e) >= m) != (e >= cut)) ++bad;
    }
}
int main() {
    std::mt19937 rng(1);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    for (int i = 0; i < 40000; ++i) look((float)exp(-80.0 * U(rng)));
    for (int i = 0; i < 40000; ++i) look((float)(0.9 * U(rng)));
    std::vector<float> at = {1.0f / 255.0f, 0.5f, 0.9f, 0.3f, 0.05f, 1.9e-35f};
    for (int k = 1; k <= 80; ++k) at.push_back((float)exp(-(double)k));
    for (int k = -3; k <= 6; ++k) at.push_back((float)exp(-ldexp(1.0, k)));
    for (float a : at)
        for (int k = -100; k <= 100; ++k) look(bits_float(float_bits(a) + (uint32_t)k));
    float cut;
    int ok = !exact_exponent_cut(0.0f, 0.99f, &cut) && !exact_exponent_cut(0.95f, 0.99f, &cut) &&
             !exact_exponent_cut(1e-36f, 0.99f, &cut) && exact_exponent_cut(0.5f, 0.3f, &cut) && cut == kInf &&
             exact_exponent_cut(0.5f, 0.5f, &cut) && cut < 0.0f;
    printf("%ld %ld %ld %d\\n", bad, none, all, ok);
}
""")
    bad, none, total, ok = map(int, out)
    assert bad == 0 and ok == 1 and total > 90_000, out
    assert none <= total // 1000   # (a matter of speed only: such a threshold's batches compare the alphas)
