// dvg_winding_fast.h -- decision-exact fast paths of the cubic winding and cubic stroke
// coverage tests.
//
// The winding contribution of a cubic segment (winding_number.h:119-157) is the sum,
// over the roots t of y(t) = pt.y that the double cubic solver (solve.h:29-64) returns,
// of [0 <= t <= 1] [x(t) - pt.x > 0] sign(y'(t)).  The reference evaluates this on
// power-basis coefficients rounded to float, so its polynomial differs from the exact
// Bezier curve by at most a few units in the last place of the coordinates.
//
// This file decides the same sum in float without the cubic solve whenever every one of
// those decisions is certain by a margin that covers that difference:
//   * the curve's y(t) - pt.y is split at its critical points; every breakpoint value
//     (ends and extrema) must be at least `ey` away from zero, so each piece crosses
//     the ray at most once, away from the piece ends (no root near t = 0 or 1, no
//     tangency);
//   * each crossing is bracketed by bisection, to 2^-6 of its piece in the screen and to
//     2^-16 in the full test (fine enough that points 1e-4 of the canvas from the curve,
//     where the edge kernel shades both sides of a boundary, are decided), and |y'| must
//     stay above a margin over the bracket, so the sign the reference computes at its root
//     is the crossing direction;
//   * x(t) - pt.x must be certainly positive or certainly negative over the bracket.
// The polynomials are evaluated on the reference's own float coefficients by Horner's rule
// with fused multiply-adds (three an evaluation).
// When any test is uncertain it returns false and the caller runs the reference's
// solve.  Host and device compile the same code (no floating-point contraction).
#pragma once

#include <cmath>

#if defined(__HIPCC__)
#define DVG_WF __host__ __device__ inline
#else
#define DVG_WF inline
#endif

namespace dvg {
namespace wf {

DVG_WF float bern3(float c0, float c1, float c2, float c3, float t) {
    float s = 1.f - t;
    return (s * s * s) * c0 + (3.f * s * s * t) * c1 + (3.f * s * t * t) * c2 + (t * t * t) * c3;
}
DVG_WF float horner3(float a, float b, float c, float d, float t) {
    return __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(a, t, b), t, c), t, d);
}
DVG_WF float rcp(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcpf(x);
#else
    return 1.f / x;
#endif
}

DVG_WF float max4(float a, float b, float c, float d) { return fmaxf(fmaxf(a, b), fmaxf(c, d)); }

// The parts of the test that depend on the segment only, computed once per segment (the
// renderer keeps them in the scene, refreshed whenever the points change).
struct CubicPrep {
    float my, mx;          // largest |y|, |x| of the control points
    float ey, ex;          // value margins' segment part, from the root accuracy of the
                           // reference's solver; ey NaN: not decidable here
    float ymin, ymax, xmax;  // control box
    float ed;              // derivative margin's segment part
    float b1, b2, y1, y2;  // interior critical points of y in (0, 1), ascending, and y there;
                           // 1 and y(1) when absent; b1 NaN: y nearly constant
    float y2max, x1max;    // |y''| and |x'| bounds
    float p0y, p3y;
    float ay, by, cy, p0x, ax, bx, cx;  // power-basis coefficients (winding_number.h:134-146)
    float pad;
};
constexpr int kPrepFloats = 24;
static_assert(sizeof(CubicPrep) == kPrepFloats * sizeof(float), "read and written as float4s");

DVG_WF CubicPrep cubic_prep(float p0x, float p0y, float p1x, float p1y, float p2x, float p2y, float p3x, float p3y) {
    CubicPrep q;
    q.my = max4(fabsf(p0y), fabsf(p1y), fabsf(p2y), fabsf(p3y));
    q.mx = max4(fabsf(p0x), fabsf(p1x), fabsf(p2x), fabsf(p3x));
    q.ymin = -max4(-p0y, -p1y, -p2y, -p3y);
    q.ymax = max4(p0y, p1y, p2y, p3y);
    q.xmax = max4(p0x, p1x, p2x, p3x);
    q.ay = -p0y + 3 * p1y - 3 * p2y + p3y;
    q.by = 3 * p0y - 6 * p1y + 3 * p2y;
    q.cy = -3 * p0y + 3 * p1y;
    q.ax = -p0x + 3 * p1x - 3 * p2x + p3x;
    q.bx = 3 * p0x - 6 * p1x + 3 * p2x;
    q.cx = -3 * p0x + 3 * p1x;
    q.p0x = p0x;
    q.p0y = p0y;
    q.p3y = p3y;
    q.pad = 0.f;
    // The reference's solver works on these float coefficients (winding_number.h:134-138).
    // Its roots are accurate to about E in t: for a near-quadratic cubic (|b| >> |a|) the
    // trigonometric branch loses precision as |b / a| grows; below |a| = 1e-6 it solves
    // the quadratic instead.
    float E = 1e-9f;
    if (!(fabsf(q.ay) < 1e-6f)) {
        const float ia = 1.f / fabsf(q.ay);
        E = 2e-7f * (fabsf(q.by) * ia + sqrtf(fabsf(q.cy) * ia) + 1.f);
    }
    // critical points of y
    const float d0 = p1y - p0y, d1 = p2y - p1y, d2 = p3y - p2y;
    const float qa = d0 - 2.f * d1 + d2, qb = 2.f * (d1 - d0), qc = d0;
    q.b1 = q.b2 = 1.f;
    // y is monotone on [0, 1] when its control differences share a strict sign (y'/3 is
    // their Bernstein combination): no interior critical point to find
    const bool mono = (d0 > 0.f && d1 > 0.f && d2 > 0.f) || (d0 < 0.f && d1 < 0.f && d2 < 0.f);
    if (!mono) {
        float r0 = -1.f, r1 = -1.f;
        const float sc = fabsf(qa) + fabsf(qb) + fabsf(qc);
        bool flat = false;
        if (fabsf(qa) > 1e-6f * sc) {
            float disc = qb * qb - 4.f * qa * qc;
            if (disc >= 0.f) {
                float sq = sqrtf(disc);
                float qq = -0.5f * (qb + (qb >= 0.f ? sq : -sq));
                r0 = qq / qa;
                r1 = qq != 0.f ? qc / qq : -1.f;
            }
        } else if (fabsf(qb) > 1e-6f * sc) {
            r0 = -qc / qb;
        } else {
            flat = true;  // y nearly constant: leave it to the solver
        }
        if (r0 > r1) {
            float tmp = r0;
            r0 = r1;
            r1 = tmp;
        }
        const bool in0 = r0 > 0.f && r0 < 1.f, in1 = r1 > 0.f && r1 < 1.f && r1 != r0;
        if (in0) q.b1 = r0;
        if (in1) (in0 ? q.b2 : q.b1) = r1;
        if (flat) q.b1 = __builtin_nanf("");
    }
    q.y1 = q.b1 == 1.f ? p3y : horner3(q.ay, q.by, q.cy, p0y, q.b1);
    q.y2 = q.b2 == 1.f ? p3y : horner3(q.ay, q.by, q.cy, p0y, q.b2);
    const float y2max = 6.f * fmaxf(fabsf(d1 - d0), fabsf(d2 - d1));  // |y''|
    q.y2max = y2max;
    const float dx0 = p1x - p0x, dx1 = p2x - p1x, dx2 = p3x - p2x;
    const float dx = fmaxf(fmaxf(fabsf(dx0), fabsf(dx1)), fabsf(dx2));
    const float dy = fmaxf(fmaxf(fabsf(d0), fabsf(d1)), fabsf(d2));
    q.x1max = 3.f * dx;  // |x'|
    q.ey = E < 1e-3f ? 3.f * E * dy : __builtin_nanf("");
    q.ex = 3.f * E * dx;
    q.ed = 1e-6f + 2.f * E * y2max;
    return q;
}

// N halvings of the bracket [lo, hi] of a root of the cubic with the given coefficients
// (rising: the cubic goes from negative to positive over the bracket).
template <int N>
DVG_WF void halve(float a, float b, float c, float d, bool rising, float &lo, float &hi) {
#pragma unroll
    for (int it = 0; it < N; it++) {
        const float mid = 0.5f * (lo + hi);
        const bool right = (horner3(a, b, c, d, mid) > 0.f) == rising;
        hi = right ? mid : hi;
        lo = right ? lo : mid;
    }
}

// Whether the crossing in [lo, hi] lies certainly right (+1) or left (-1) of the point, y'
// keeping the crossing's sign with margin ed, else 0.  The true crossing of any ray height
// within hv of the evaluated one (rounding, and the spread of heights decided at once) lies
// up to hv / min |y'| outside the bracket: the bracket grows by 2 hv / |y'(m)|, and |y'| must
// stay above half of |y'(m)| over it.
DVG_WF int crossing_side(const CubicPrep &q, float ptx, bool rising, float lo, float hi, float ed, float ex, float hv) {
    const float m = 0.5f * (lo + hi);
    const float yd = __builtin_fmaf(__builtin_fmaf(3.f * q.ay, m, 2.f * q.by), m, q.cy), a = fabsf(yd);
    const float half = __builtin_fmaf(2.03f * hv, rcp(a), 0.5f * (hi - lo));
    const float low = __builtin_fmaf(-q.y2max, half, a);
    const float xm = horner3(q.ax, q.bx, q.cx, q.p0x, m) - ptx, xv = __builtin_fmaf(q.x1max, half, ex);
    if ((yd > 0.f) != rising || !(low >= 0.5f * a) || !(low > ed)) return 0;
    return xm > xv ? 1 : (xm < -xv ? -1 : 0);
}

// Returns true and sets `w` when the contribution is decided.  With hx, hy > 0 it decides for
// every point within hx, hy of (ptx, pty) at once (the two sides of a boundary sample): every
// margin grows by that much.  FULL = false stops at 6 halvings of a crossing's piece (the
// screen of dvg_wave.h: what is open then is a few per cent, cheaper to gather and refine
// together than to refine beside lanes that are done).
template <bool FULL>
DVG_WF bool cubic_winding_test(const CubicPrep &q, float ptx, float pty, int &w, float hx = 0.f, float hy = 0.f) {
    const float M = fmaxf(q.my, fabsf(pty) + hy) + 1.f;
    const float Mx = fmaxf(q.mx, fabsf(ptx) + hx) + 1.f;
    // value margins: the reference's coefficients are within ~2e-6 M of the curve's, and
    // its roots within E of the true ones
    const float ey = __builtin_fmaf(1e-5f, M, q.ey) + hy;
    const float ex = __builtin_fmaf(1e-5f, Mx, q.ex) + hx;
    w = 0;
    if (!(ey == ey)) return false;
    // hull above or below the ray, or entirely left of the point: every root has x(t) < pt.x
    if (q.ymin - pty > ey || q.ymax - pty < -ey || q.xmax < ptx - ex) return true;
    // values at the breakpoints 0, b1, b2, 1; b1 NaN (y nearly constant) makes y1 NaN
    const float f0 = q.p0y - pty, f1 = q.y1 - pty, f2 = q.y2 - pty, f3 = q.p3y - pty;
    if (!(fabsf(f0) > ey && fabsf(f1) > ey && fabsf(f2) > ey && fabsf(f3) > ey)) return false;
    const float ed = __builtin_fmaf(3e-4f, M, q.ed);  // derivative margin
    const float hv = __builtin_fmaf(2e-6f, M, hy);    // rounding of the evaluated heights
    const bool s0 = f0 > 0.f, s1 = f1 > 0.f, s2 = f2 > 0.f, s3 = f3 > 0.f;
    bool c1 = s0 != s1, c2 = s1 != s2, c3 = s2 != s3;
    int acc = 0;
    // one crossing a turn, whichever piece it is in
#pragma nounroll
    while (c1 || c2 || c3) {
        float lo = c1 ? 0.f : (c2 ? q.b1 : q.b2), hi = c1 ? q.b1 : (c2 ? q.b2 : 1.f);
        const bool rising = c1 ? s1 : (c2 ? s2 : s3);
        c3 = c3 && (c1 || c2);
        c2 = c2 && c1;
        c1 = false;
        halve<6>(q.ay, q.by, q.cy, f0, rising, lo, hi);
        int xs = crossing_side(q, ptx, rising, lo, hi, ed, ex, hv);
        if (FULL && xs == 0) {
            halve<10>(q.ay, q.by, q.cy, f0, rising, lo, hi);
            xs = crossing_side(q, ptx, rising, lo, hi, ed, ex, hv);
        }
        if (xs == 0) return false;
        if (xs > 0) acc += rising ? 1 : -1;
    }
    w = acc;
    return true;
}

// Returns true and sets `w` when the contribution is decided.
DVG_WF bool cubic_winding_fast(float p0x, float p0y, float p1x, float p1y, float p2x, float p2y, float p3x,
                               float p3y, float ptx, float pty, int &w) {
    return cubic_winding_test<true>(cubic_prep(p0x, p0y, p1x, p1y, p2x, p2y, p3x, p3y), ptx, pty, w);
}

// Stroke coverage of a cubic segment (within_distance.h:119-272) accepts only when one
// of the curve points it evaluates (the ends and the stationary points of the distance)
// is closer than the stroke radius.  The test below holds when every point of the curve is
// at least rmax + a rounding margin away from pt, so that test certainly rejects: the
// curve lies within (h^2 / 8) max|B''| of its chords over 8 equal steps of t, with
// |B''| <= 6 max|second differences of the control points| per coordinate.
// The segment-only part: the nine polyline points at t = k/8 (the ends of the curve among
// them), one over each chord's squared length (0 for a chord of no length), the largest
// control-point coordinate magnitude `mc` and the chords' deviation bound `dev`.
struct StrokePrep {
    float x[9], y[9], inv[8];
    float mc, dev;
};
constexpr int kStrokeFloats = 28;
static_assert(sizeof(StrokePrep) == kStrokeFloats * sizeof(float), "read and written as float4s");

DVG_WF StrokePrep stroke_prep(float p0x, float p0y, float p1x, float p1y, float p2x, float p2y, float p3x, float p3y) {
    StrokePrep q;
    q.mc = fmaxf(max4(fabsf(p0x), fabsf(p1x), fabsf(p2x), fabsf(p3x)), max4(fabsf(p0y), fabsf(p1y), fabsf(p2y), fabsf(p3y)));
    const float sx = fmaxf(fabsf(p0x - 2.f * p1x + p2x), fabsf(p1x - 2.f * p2x + p3x));
    const float sy = fmaxf(fabsf(p0y - 2.f * p1y + p2y), fabsf(p1y - 2.f * p2y + p3y));
    q.dev = (6.f / 512.f) * sqrtf(sx * sx + sy * sy) * 1.001f;
#pragma unroll
    for (int k = 0; k <= 8; k++) {
        const float t = 0.125f * (float)k;
        q.x[k] = k == 0 ? p0x : (k == 8 ? p3x : bern3(p0x, p1x, p2x, p3x, t));
        q.y[k] = k == 0 ? p0y : (k == 8 ? p3y : bern3(p0y, p1y, p2y, p3y, t));
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const float dx = q.x[k + 1] - q.x[k], dy = q.y[k + 1] - q.y[k], l2 = dx * dx + dy * dy;
        q.inv[k] = l2 > 1e-30f ? 1.f / l2 : 0.f;
    }
    return q;
}

// The test itself: the distance from pt to each chord at the clamped projection.  (A rounded
// projection parameter overstates a chord's distance by far less than the margin.)
DVG_WF bool stroke_farther(const StrokePrep &q, float ptx, float pty, float rmax) {
    const float M = fmaxf(q.mc, fmaxf(fabsf(ptx), fabsf(pty))) + 1.f;
    const float need = rmax + 1e-4f * M + q.dev, n2 = need * need;
    bool far = true;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const float dx = q.x[k + 1] - q.x[k], dy = q.y[k + 1] - q.y[k], wx = ptx - q.x[k], wy = pty - q.y[k];
        const float t = fminf(fmaxf(__builtin_fmaf(wx, dx, wy * dy) * q.inv[k], 0.f), 1.f);
        const float ex = __builtin_fmaf(-t, dx, wx), ey = __builtin_fmaf(-t, dy, wy);
        far = far && __builtin_fmaf(ex, ex, ey * ey) > n2;
    }
    return far;
}

// Every point within `reach` of pt lies within the stroke's radius (r0, r3) of one and the same end
// of the curve, with a margin for rounding (the other half of a decision for a whole box).
DVG_WF bool stroke_ends_within(const StrokePrep &q, float ptx, float pty, float r0, float r3, float reach) {
    const float less = reach + 1e-4f * (fmaxf(q.mc, fmaxf(fabsf(ptx), fabsf(pty))) + 1.f);
    const float c0 = r0 - less, c3 = r3 - less;
    const float ux = ptx - q.x[0], uy = pty - q.y[0], vx = ptx - q.x[8], vy = pty - q.y[8];
    return (c0 > 0.f && ux * ux + uy * uy < c0 * c0) || (c3 > 0.f && vx * vx + vy * vy < c3 * c3);
}

DVG_WF bool cubic_certainly_farther(float p0x, float p0y, float p1x, float p1y, float p2x, float p2y, float p3x,
                                    float p3y, float ptx, float pty, float rmax) {
    return stroke_farther(stroke_prep(p0x, p0y, p1x, p1y, p2x, p2y, p3x, p3y), ptx, pty, rmax);
}

}  // namespace wf
}  // namespace dvg
