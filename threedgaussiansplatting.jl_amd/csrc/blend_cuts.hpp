// blend_cuts.hpp — where blending may leave an entry out: the exponents that stand for min_alpha (host),
// and the box around a Gaussian's mean outside which no alpha reaches it.
#pragma once

#include <cmath>

#include "tdgs_math.hpp"

namespace tdgs {

// Exponent below which blending can skip an entry: for e < exponent_cut(min_alpha),
// exp_f(e) (relative error a few 1e-7) is below min_alpha, so alpha < min_alpha. A margin of
// 1e-3 in the exponent covers the rounding; no cut without a positive min_alpha.
inline float exponent_cut(float min_alpha) {
    if (!(min_alpha > 0.0f)) return -__builtin_inff();
    return std::nextafter((float)(std::log((double)min_alpha) - 1e-3), -__builtin_inff());
}

// The exponent from which alpha = min(exp_f(e), max_alpha) reaches min_alpha: alpha >= min_alpha exactly for
// e >= *cut (infinity where max_alpha stays below min_alpha). exp_f is within 0.91 ulp (1.1e-7 relative) of exp, so only
// exponents within 1.1e-7 of log(min_alpha) are in doubt: two floats to either side where the exponents are at least 1
// in size (1.2e-7 apart or more), looked for within four; 15 up to a min_alpha of 0.9 (7.4e-9 apart), looked for within
// 32. The switch among them has to be a clean one (above a min_alpha of 1/e several neighbouring exponents share
// an alpha, and exp_f may step back by an ulp). (Each look costs the host ~40 ns, which a frame with host counts waits for.) False when there is
// none, or when *cut < -80 (results of exp_f near its flush to zero).
inline bool exact_exponent_cut(float min_alpha, float max_alpha, float* cut) {
    *cut = __builtin_inff();
    if (max_alpha < min_alpha) return true;
    if (!(min_alpha > 0.0f) || !(min_alpha <= 0.9f) || !(max_alpha >= min_alpha)) return false;
    const float mid = (float)std::log((double)min_alpha);   // negative: one float up is one less in the bits
    if (!(mid >= -80.0f)) return false;
    const int span = mid <= -1.0f ? 4 : 32;
    bool reached = false;
    for (int k = -span; k < span; ++k) {
        const float e = bits_float(float_bits(mid) - (uint32_t)k);
        const bool r = exp_f(e) >= min_alpha;
        if (r ? k == -span : reached) return false;
        if (r && !reached) *cut = e;
        reached = r;
    }
    return reached;
}

// The half sides (r_x, r_y) of a box around the mean outside which x < cut, for x = fl(-(p du^2 + q du dv +
// s dv^2)), p = -A, q = -B, s = -C > 0: x = cut is an ellipse whose du reaches sqrt(-cut s / det), det =
// p s - q^2 / 4, there at dv = -q du / (2 s). Each of the five roundings of x is off by at most 2^-24 of a term of at
// most 2 p du^2, 5 2^-24 p du^2 in all (to first order the same elsewhere outside the box), which equals
// 3e-7 (p s / det) of cut on the ellipse: det less 1e-6 p s covers it, for needles of any length. The
// determinant is formed in double (p s and q^2 / 4 agree to 1 in 1e4 and more), the box widened by 1e-4 of its size and
// 1e-2 pixels for the rounding of du, dv, the cut and the square root. No bound (infinite sides) where no positive
// determinant is left or anything is NaN, none at all (negative sides) where a positive cut says that no alpha
// reaches min_alpha. The cut's own margin (1e-3) covers its error.
TDGS_HD void cut_box(float A, float B, float C, float cut, float* rx, float* ry) {
    const float p = -A, s = -C;
    const double det = (1.0 - 1e-6) * ((double)p * s) - 0.25 * (double)B * B;
    const float k = -cut / (float)det;
    const float x2 = k * s, y2 = k * p;
    const bool bounded = p > 0.0f && s > 0.0f && det > 0.0 && x2 >= 0.0f && y2 >= 0.0f && x2 < kInf && y2 < kInf;
    *rx = bounded ? fmaf(sqrtf(x2), 1.0001f, 0.01f) : kInf;
    *ry = bounded ? fmaf(sqrtf(y2), 1.0001f, 0.01f) : kInf;
    if (cut > 1e-3f) *rx = *ry = -kInf;
}

}  // namespace tdgs
