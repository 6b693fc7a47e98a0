// dvg_quintic.h -- double-precision roots: quadratic, cubic, and the stationary points of the
// distance from a point to a cubic segment.
//
// Host and device compile the same code (no floating-point contraction), so that the searches
// can be compared with the reference's arithmetic on the CPU.
#pragma once

#include <cmath>
#include <cstdint>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define DVG_Q __host__ __device__ __forceinline__
#else
#define DVG_Q inline
#endif

#include "dvg_crmath.h"

namespace dvg {

constexpr double kPi = 3.14159265358979323846;

// Roots of a t^2 + b t + c, ascending (solve.h:8-27)
DVG_Q bool solve_quadratic_d(double a, double b, double c, double *t0, double *t1) {
    double discrim = b * b - 4 * a * c;
    if (discrim < 0) return false;
    double root_discrim = __builtin_sqrt(discrim);
    double q = b < 0 ? -0.5f * (b - root_discrim) : -0.5f * (b + root_discrim);
    double r0 = q / a, r1 = c / q;
    if (r0 > r1) {
        double tmp = r0;
        r0 = r1;
        r1 = tmp;
    }
    *t0 = r0;
    *t1 = r1;
    return true;
}

// solve_cubic<double> (solve.h:29-64).  CR selects the correctly rounded acos, cos and
// pow; the default uses the device libm.
template <bool CR = false>
DVG_Q int solve_cubic_d(double a, double b, double c, double d, double t[3]) {
    if (fabs(a) < 1e-6f) {
        if (solve_quadratic_d(b, c, d, &t[0], &t[1])) return 2;
        return 0;
    }
    b /= a;
    c /= a;
    d /= a;
    double Q = (b * b - 3 * c) / 9.f;
    double R = (2 * b * b * b - 9 * b * c + 27 * d) / 54.f;
    if (R * R < Q * Q * Q) {
        double x = R / sqrt(Q * Q * Q);
        double theta = CR ? cr::acos_cr(x) : acos(x);
        double sq = sqrt(Q);
        double a0 = theta / 3.f, a1 = (theta + 2.f * kPi) / 3.f, a2 = (theta - 2.f * kPi) / 3.f;
        t[0] = -2.f * sq * (CR ? cr::cos_cr(a0) : cos(a0)) - b / 3.f;
        t[1] = -2.f * sq * (CR ? cr::cos_cr(a1) : cos(a1)) - b / 3.f;
        t[2] = -2.f * sq * (CR ? cr::cos_cr(a2) : cos(a2)) - b / 3.f;
        return 3;
    } else {
        double base = R > 0 ? R + sqrt(R * R - Q * Q * Q) : -R + sqrt(R * R - Q * Q * Q);
        double root = CR ? cr::pow_cr(base, 1. / 3.) : pow(base, 1. / 3.);
        double A = R > 0 ? -root : root;
        double B = fabs(A) > 1e-6f ? Q / A : 0.0;
        t[0] = (A + B) - b / 3.0;
        return 1;
    }
}

// The stationary points of the distance to a cubic: roots of a quintic, isolated by the roots
// of a cubic and a linear factor (within_distance.h:119-272, compute_distance.h:127-280).  The
// arithmetic is double; next to the reference's, divisions by one number are products with
// its reciprocal, polynomials are evaluated by Horner's rule with fused multiply-adds and the
// trigonometric roots come from one sine and cosine: roundings of the last bit or two, in
// interval ends and iterates that are then stored as floats.  (A point's coverage by its 2,048
// strokes took half of the edge kernel: 17 double divisions, three cosines, a power and 45
// double operations a Newton step for each.)
//
// Whether the reference finds a root, so perhaps the closest point at all, can hang on those last
// bits, and then its own operations are used (quintic_search_plain):
//   * where the normalised coefficients are large (kQuinticLarge).  The curve is nearly a quadratic
//     or a line -- a quadratic written as a cubic has coefficients of 1e9 to 1e17, made of the
//     rounding of its float coordinates -- and the interval ends are rounding too.  1.4e-4 of the
//     points near such strokes were covered otherwise; none in 4 million up to coefficients of 1e7;
//   * where the quintic at an interval end is zero to rounding, or the cubic's roots are double
//     (kQuinticOpen): curves through points A and B only, as A B B B (handles on an end), have
//     multiple roots in both polynomials.  2.9e-3 of the points near A B B B were covered
//     otherwise.  Of ordinary curves 3e-5 of the points come here.
// With both, no decision differs over 30 million cases of 30 families of curves.  Looking for them
// costs 2% of a pass over 2,048 strokes and 5% of a distance field; 300 strokes of three
// quadratics written as cubics at 256x256, 4 samples, take 0.21 ms forward and 0.43 backward
// instead of 0.14 and 0.30.
struct Quintic {
    double A, B, C, D, E, F;  // leading coefficient, and the others divided by it
};
// The quintic's coefficients before the division by the leading one, formed in float as the
// reference does (within_distance.h:174-187)
struct QuinticSums {
    float A, B, C, D, E, F;
};
DVG_Q QuinticSums cubic_quintic_sums(float p0x, float p0y, float p1x, float p1y, float p2x, float p2y, float p3x,
                                     float p3y, float ptx, float pty) {
    const float ax = -p0x + 3 * p1x - 3 * p2x + p3x, ay = -p0y + 3 * p1y - 3 * p2y + p3y;
    const float bx = 3 * p0x - 6 * p1x + 3 * p2x, by = 3 * p0y - 6 * p1y + 3 * p2y;
    const float cx = -3 * p0x + 3 * p1x, cy = -3 * p0y + 3 * p1y;
    const float dx = p0x - ptx, dy = p0y - pty;
    QuinticSums q;
    q.A = 3 * (ax * ax + ay * ay);
    q.B = 5 * (ax * bx + ay * by);
    q.C = 4 * (ax * cx + ay * cy) + 2 * (bx * bx + by * by);
    q.D = 3 * ((bx * cx + by * cy) + (ax * dx + ay * dy));
    q.E = (cx * cx + cy * cy) + 2 * (dx * bx + dy * by);
    q.F = dx * cx + dy * cy;
    return q;
}
DVG_Q Quintic cubic_quintic(const QuinticSums &u) {
    const double A = u.A, inv = 1.0 / A;
    return Quintic{A, u.B * inv, u.C * inv, u.D * inv, u.E * inv, u.F * inv};
}
constexpr float kQuinticLarge = 1e6f;
constexpr float kQuinticOpen = 1e-9f;
// What tells that the roots of a quintic hang on rounding, from its sums: the sum of the
// coefficients' magnitudes and whether the derivative vanishes at 1 beside it.
struct QuinticScale {
    float size;
    bool flat_end;
    DVG_Q bool large(float A) const { return !(size < kQuinticLarge * A); }  // also for A = 0, not a number
};
DVG_Q QuinticScale quintic_scale(const QuinticSums &u) {
    const float size = u.A + (fabsf(u.B) + fabsf(u.C)) + (fabsf(u.D) + fabsf(u.E)) + fabsf(u.F);
    return QuinticScale{size, fabsf(5 * u.A + 4 * u.B + 3 * u.C + 2 * u.D + u.E) < 1e-4f * size};
}
DVG_Q double quintic_eval(const Quintic &q, double t) {
    return __builtin_fma(__builtin_fma(__builtin_fma(__builtin_fma(t + q.B, t, q.C), t, q.D), t, q.E), t, q.F);
}
DVG_Q double quintic_deriv(const Quintic &q, double t) {
    return __builtin_fma(__builtin_fma(__builtin_fma(__builtin_fma(5.0, t, 4 * q.B), t, 3 * q.C), t, 2 * q.D), t, q.E);
}
// sin and cos of x in [0, pi / 3] by their Taylor series (to x^21 and x^20; the next terms are
// below 1e-20)
DVG_Q void sincos_third(double x, double &s, double &c) {
    const double z = x * x;
    double p = 1.0 / 51090942171709440000.0, r = 1.0 / 2432902008176640000.0;
    p = __builtin_fma(p, z, -1.0 / 121645100408832000.0);
    r = __builtin_fma(r, z, -1.0 / 6402373705728000.0);
    p = __builtin_fma(p, z, 1.0 / 355687428096000.0);
    r = __builtin_fma(r, z, 1.0 / 20922789888000.0);
    p = __builtin_fma(p, z, -1.0 / 1307674368000.0);
    r = __builtin_fma(r, z, -1.0 / 87178291200.0);
    p = __builtin_fma(p, z, 1.0 / 6227020800.0);
    r = __builtin_fma(r, z, 1.0 / 479001600.0);
    p = __builtin_fma(p, z, -1.0 / 39916800.0);
    r = __builtin_fma(r, z, -1.0 / 3628800.0);
    p = __builtin_fma(p, z, 1.0 / 362880.0);
    r = __builtin_fma(r, z, 1.0 / 40320.0);
    p = __builtin_fma(p, z, -1.0 / 5040.0);
    r = __builtin_fma(r, z, -1.0 / 720.0);
    p = __builtin_fma(p, z, 1.0 / 120.0);
    r = __builtin_fma(r, z, 1.0 / 24.0);
    p = __builtin_fma(p, z, -1.0 / 6.0);
    r = __builtin_fma(r, z, -0.5);
    s = __builtin_fma(p * z, x, x);
    c = __builtin_fma(r, z, 1.0);
}
// Roots of a t^3 + b t^2 + c t + d as solve_cubic_d returns them (solve.h:29-64).  `open` is set
// when two of them are so close that the number found hangs on rounding.
DVG_Q int isolating_cubic(double a, double b, double c, double d, double (&t)[3], bool &open) {
    if (fabs(a) < 1e-6f) {
        open = !(fabs(c * c - 4 * b * d) > kQuinticOpen * (c * c));
        return solve_quadratic_d(b, c, d, &t[0], &t[1]) ? 2 : 0;
    }
    const double inv = 1.0 / a, third = 1.0 / 3.0;
    b *= inv;
    c *= inv;
    d *= inv;
    const double Q = (b * b - 3 * c) * (1.0 / 9.0);
    const double R = (2 * b * b * b - 9 * b * c + 27 * d) * (1.0 / 54.0);
    const double Q3 = Q * Q * Q, R2 = R * R, b3 = b * third;
    open = !(fabs(R2 - Q3) > kQuinticOpen * R2);
    if (R2 < Q3) {
        double s, co;
        sincos_third(acos(R / sqrt(Q3)) * third, s, co);
        const double h = 0.86602540378443864676 * s, m = -2.0 * __builtin_sqrt(Q);
        t[0] = m * co - b3;
        t[1] = m * (-0.5 * co - h) - b3;
        t[2] = m * (-0.5 * co + h) - b3;
        return 3;
    }
    const double root = cbrt(fabs(R) + __builtin_sqrt(R2 - Q3));
    const double A = R > 0 ? -root : root;
    const double B = fabs(A) > 1e-6f ? Q / A : 0.0;
    t[0] = (A + B) - b3;
    return 1;
}
// The interval ends in ascending order: the linear factor's root if it is in [0, 1], and the
// first num_sol of pr; returns their number.  The reference's uninitialised intervals[0]
// (isolator root outside [0, 1]) is treated as absent.  All indices are compile-time constants
// (slots past the number are not read as such), so the array stays in registers.
DVG_Q int sort_intervals(bool first, float q_root, int num_sol, const double (&pr)[3], float (&iv)[4]) {
    const int n = num_sol + (first ? 1 : 0);
    iv[0] = first ? q_root : (float)pr[0];
    iv[1] = first ? (float)pr[0] : (float)pr[1];
    iv[2] = first ? (float)pr[1] : (float)pr[2];
    iv[3] = (float)pr[2];
    // insertion sort of the first n
#pragma unroll
    for (int j = 1; j < 4; j++) {
        bool go = j < n;
#pragma unroll
        for (int k = j; k > 0; k--) {
            go = go && iv[k - 1] > iv[k];
            const float lo = go ? iv[k] : iv[k - 1], hi = go ? iv[k - 1] : iv[k];
            iv[k - 1] = lo;
            iv[k] = hi;
        }
    }
    return n;
}
// Isolating intervals (within_distance.h:195-216)
DVG_Q int quintic_intervals(const Quintic &q, float (&iv)[4], bool &open) {
    // the reference's float fractions
    const double p1A = (2 / 5.f) * q.C - (4 / 25.f) * q.B * q.B;
    const double p1B = (3 / 5.f) * q.D - (3 / 25.f) * q.B * q.C;
    const double p1C = (4 / 5.f) * q.E - (2 / 25.f) * q.B * q.D;
    const double p1D = q.F - q.B * q.E * (1.0 / 25.0);
    const double q_root = q.B * -0.2;
    double pr[3] = {0.0, 0.0, 0.0};
    const int num_sol = isolating_cubic(p1A, p1B, p1C, p1D, pr, open);
    return sort_intervals(q_root >= 0 && q_root <= 1, (float)q_root, num_sol, pr, iv);
}
// A first reciprocal, correct to about a float's precision
DVG_Q double quintic_rcp(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcp(x);
#else
    return (1.0 / x) * (1.0 + 6e-8);
#endif
}
// Newton's iteration kept in its bracket (within_distance.h:232-262)
DVG_Q float quintic_root(const Quintic &q, float lb, float ub) {
    float t = 0.5f * (lb + ub);
#pragma nounroll
    for (int it = 0; it < 20; it++) {
        if (!(t >= lb && t <= ub)) t = 0.5f * (lb + ub);
        const double td = t;
        const double value = quintic_eval(q, td);
        if (fabs(value) < 1e-5f || it == 19) break;
        if (value > 0.f)
            ub = t;
        else
            lb = t;
        const double deriv = quintic_deriv(q, td);
        double r = quintic_rcp(deriv);
        r = __builtin_fma(__builtin_fma(-deriv, r, 1.0), r, r);
        r = __builtin_fma(__builtin_fma(-deriv, r, 1.0), r, r);
        t = (float)__builtin_fma(-value, r, td);
    }
    return t;
}
// |x| by its upper half: enough to compare magnitudes, in one register
DVG_Q uint32_t high_word(double x) {
    uint64_t v;
    __builtin_memcpy(&v, &x, sizeof(v));
    return (uint32_t)(v >> 32) & 0x7fffffffu;
}
// Calls visit(t) for the root in each interval with a sign change, in order, until it
// returns true.  The brackets are found first, so that the lanes of a wave run their first
// searches together, then their second ones, whichever intervals those are.  False, and nothing
// visited, when the signs at the interval ends hang on rounding.
template <class Visit>
DVG_Q bool quintic_search(const Quintic &q, const QuinticScale &scale, const Visit &visit) {
    float iv[4];
    bool open = false;
    const int n = quintic_intervals(q, iv, open);
    const uint32_t small = high_word((double)(kQuinticOpen * scale.size) * (1.0 / q.A));
    unsigned found = 0, falls = 0;  // intervals with a sign change, and those where it is downward
    double at_lower = quintic_eval(q, 0.0);
    bool more = true;
#pragma unroll
    for (int j = 0; j < 5; j++) {
        const bool inner = j < 4 && j < n;
        const float end = j < 4 ? iv[j < 4 ? j : 3] : 1.f;
        const bool use = more && j <= n && !(inner && end < 0.f);
        const float upper = inner ? (end < 1.f ? end : 1.f) : 1.f;
        const double at_upper = quintic_eval(q, upper);
        // at 1 a root of its own does no harm (a handle of no length has one)
        const bool counts = j < 4 ? inner && end > -1e-5f && end < 1.00001f : scale.flat_end;
        open = open || (counts && high_word(at_upper) < small);
        const bool change = use && !(at_lower * at_upper > 0);
        if (at_lower > at_upper) falls |= 1u << j;
        if (change) {
            found |= 1u << j;
            more = !(upper >= 1.f);
            at_lower = at_upper;
        }
    }
    if (open) return false;
    float lower = 0.f;
#pragma nounroll
    while (found) {
        const int j = __builtin_ctz(found);
        found &= found - 1;
        const float end = j < 2 ? (j == 0 ? iv[0] : iv[1]) : (j == 2 ? iv[2] : iv[3]);
        const float upper = j < 4 && j < n && end < 1.f ? end : 1.f;
        const bool down = (falls >> j) & 1u;
        const float lb = down ? upper : lower, ub = down ? lower : upper;
        lower = upper;
        if (visit(quintic_root(q, lb, ub))) break;
    }
    return true;
}

// The same with the reference's operations in the reference's order (within_distance.h:187-262)
DVG_Q double quintic_eval_plain(const Quintic &q, double t) {
    return t * t * t * t * t + q.B * t * t * t * t + q.C * t * t * t + q.D * t * t + q.E * t + q.F;
}
DVG_Q double quintic_deriv_plain(const Quintic &q, double t) {
    return 5 * t * t * t * t + 4 * q.B * t * t * t + 3 * q.C * t * t + 2 * q.D * t + q.E;
}
DVG_Q Quintic cubic_quintic_plain(const QuinticSums &u) {
    const double A = u.A;
    return Quintic{A, u.B / A, u.C / A, u.D / A, u.E / A, u.F / A};
}
DVG_Q int quintic_intervals_plain(const Quintic &q, float (&iv)[4]) {
    double pr[3] = {0.0, 0.0, 0.0};
    const int num_sol = solve_cubic_d((2 / 5.f) * q.C - (4 / 25.f) * q.B * q.B, (3 / 5.f) * q.D - (3 / 25.f) * q.B * q.C,
                                      (4 / 5.f) * q.E - (2 / 25.f) * q.B * q.D, q.F - q.B * q.E / 25.f, pr);
    const double q_root = -q.B / 5.f;
    return sort_intervals(q_root >= 0 && q_root <= 1, (float)q_root, num_sol, pr, iv);
}
template <class Visit>
DVG_Q void quintic_search_plain(const Quintic &q, const float (&iv)[4], int n, const Visit &visit) {
    float lower = 0.f;
#pragma nounroll
    for (int j = 0; j < n + 1; j++) {
        const float end = j == 0 ? iv[0] : (j == 1 ? iv[1] : (j == 2 ? iv[2] : iv[3]));
        if (j < n && end < 0.f) continue;
        const float upper = j < n ? (end < 1.f ? end : 1.f) : 1.f;
        const double at_lower = quintic_eval_plain(q, lower), at_upper = quintic_eval_plain(q, upper);
        if (at_lower * at_upper > 0) continue;
        float lb = at_lower > at_upper ? upper : lower, ub = at_lower > at_upper ? lower : upper;
        float t = 0.5f * (lb + ub);
#pragma nounroll
        for (int it = 0; it < 20; it++) {
            if (!(t >= lb && t <= ub)) t = 0.5f * (lb + ub);
            const double td = t, value = quintic_eval_plain(q, td);
            if (fabs(value) < 1e-5f || it == 19) break;
            if (value > 0.f)
                ub = t;
            else
                lb = t;
            t = (float)(td - value / quintic_deriv_plain(q, td));
        }
        if (visit(t) || upper >= 1.f) break;
        lower = upper;
    }
}

}  // namespace dvg
