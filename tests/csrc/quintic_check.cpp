// Compares the renderer's closest points of cubic segments (diffvg_amd/csrc/dvg_quintic.h) with
// the oracle's restatement of the reference's searches (oracle/orc_query.h,
// within_distance.h:174-262).  Test infrastructure only.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <random>

#include "../../diffvg_amd/csrc/dvg_quintic.h"
#include "../../oracle/orc_query.h"

namespace orc {
thread_local Counters *g_tc = nullptr;
thread_local bool t_q8_slot = false;
}  // namespace orc

namespace {
using orc::V2;

float at(const V2 *p, V2 pt, float t) { return orc::dist_sq(orc::ceval(p[0], p[1], p[2], p[3], t), pt); }

// Smallest distance over the ends and the points the reference's search visits.
float reference_distance(const V2 *p, V2 pt) {
    float best = std::min(at(p, pt, 0.f), at(p, pt, 1.f));
    const orc::Quintic q = orc::cubic_quintic(p[0], p[1], p[2], p[3], pt);
    float iv[4], lower = 0.f;
    const int n = orc::quintic_intervals(q, iv);
    for (int j = 0; j < n + 1; j++) {
        if (j < n && iv[j] < 0.f) continue;
        const float upper = j < n ? orc::fmin_r(iv[j], 1.f) : 1.f;
        const double a = orc::quintic_eval(q, lower), b = orc::quintic_eval(q, upper);
        if (a * b > 0) continue;
        best = std::fmin(best, at(p, pt, a > b ? orc::quintic_root(q, upper, lower) : orc::quintic_root(q, lower, upper)));
        if (upper >= 1.f) break;
        lower = upper;
    }
    return std::sqrt(best);
}

// The same as the kernels do it (cubic_stroke_search, cubic_closest).
float renderer_distance(const V2 *p, V2 pt, int64_t &large) {
    using namespace dvg;
    float best = std::min(at(p, pt, 0.f), at(p, pt, 1.f));
    const QuinticSums u =
        cubic_quintic_sums(p[0].x, p[0].y, p[1].x, p[1].y, p[2].x, p[2].y, p[3].x, p[3].y, pt.x, pt.y);
    const auto visit = [&](float t) {
        best = std::fmin(best, at(p, pt, t));
        return false;
    };
    const QuinticScale scale = quintic_scale(u);
    if (scale.large(u.A) || !quintic_search(cubic_quintic(u), scale, visit)) {
        const Quintic v = cubic_quintic_plain(u);
        float iv[4];
        const int n = quintic_intervals_plain(v, iv);
        quintic_search_plain(v, iv, n, visit);
        large++;
    }
    return std::sqrt(best);
}
}  // namespace

extern "C" {
// mode 0: random; 1: straight, control points at thirds; 2: a quadratic written as a cubic;
// 3: first handle of no length; 4: both handles of no length; 5: closed loop; 6: horizontal; 7:
// large coordinates; 8: tiny; 9: a quadratic written as a cubic and moved by 1e-6 to 1; 10: an
// arc as four-point circles have it, on whole coordinates, and its centre; 11 to 15: with points
// A and B only, A A A B, A B B B, A B A B, A B B A and one point; 16: second handle of no length.
// Half of the points lie about one stroke radius from the curve.  out: cases, cases that take
// the plain search, cases whose distances differ by more than 1e-3, cases that a stroke of that
// radius covers in one but not in the other; worst: the largest difference of the distances.
void quintic_fuzz(int mode, int64_t n, uint64_t seed, int64_t *out, float *worst) {
    std::mt19937_64 g(seed);
    std::uniform_real_distribution<float> U(0.f, 1.f);
    std::normal_distribution<float> N(0.f, 1.f);
    int64_t large = 0, far = 0, flips = 0;
    *worst = 0.f;
    for (int64_t i = 0; i < n; i++) {
        const float cx = 500.f * U(g), cy = 500.f * U(g), sp = 0.5f + 20.f * U(g), r = 0.5f + 3.5f * U(g);
        V2 p[4];
        for (V2 &x : p) x = V2{cx + sp * N(g), cy + sp * N(g)};
        if (mode == 1)
            for (int k = 1; k < 3; k++)
                p[k] = V2{p[0].x + (p[3].x - p[0].x) * (float)k / 3.f, p[0].y + (p[3].y - p[0].y) * (float)k / 3.f};
        if (mode == 2 || mode == 9) {
            const float e = mode == 9 ? std::pow(10.f, -6.f + 6.f * U(g)) : 0.f;
            const V2 c = p[1];
            p[1] = V2{(p[0].x + 2 * c.x) / 3 + e * N(g), (p[0].y + 2 * c.y) / 3 + e * N(g)};
            p[2] = V2{(p[3].x + 2 * c.x) / 3 + e * N(g), (p[3].y + 2 * c.y) / 3 + e * N(g)};
        }
        if (mode == 3 || mode == 4) p[1] = p[0];
        if (mode == 4) p[2] = p[3];
        if (mode == 5) p[3] = p[0];
        if (mode >= 11 && mode <= 15) {
            static const int order[5][4] = {{0, 0, 0, 1}, {0, 1, 1, 1}, {0, 1, 0, 1}, {0, 1, 1, 0}, {0, 0, 0, 0}};
            const V2 ab[2] = {p[0], p[3]};
            for (int k = 0; k < 4; k++) p[k] = ab[order[mode - 11][k]];
        }
        if (mode == 16) p[2] = p[3];
        for (V2 &x : p) {
            if (mode == 6) x = V2{cx + 3.f * (x.x - cx), cy};
            if (mode == 7) x = V2{40.f * x.x, 40.f * x.y};
            if (mode == 8) x = V2{cx + 0.002f * (x.x - cx), cy + 0.002f * (x.y - cy)};
        }
        const float R = std::floor(1.f + 30.f * U(g)), X = std::floor(cx), Y = std::floor(cy);
        if (mode == 10) {
            p[0] = V2{X + R, Y};
            p[1] = V2{X + R, Y + 0.5522847f * R};
            p[2] = V2{X + 0.5522847f * R, Y + R};
            p[3] = V2{X, Y + R};
        }
        const V2 c = orc::ceval(p[0], p[1], p[2], p[3], U(g));
        const float a = 6.2831853f * U(g), rr = (mode == 8 ? 0.01f : 1.f) * r * (0.8f + 0.4f * U(g));
        V2 pt{c.x + rr * std::cos(a), c.y + rr * std::sin(a)};
        if (i & 1) pt = V2{c.x + sp * N(g), c.y + sp * N(g)};
        if (mode == 10 && (i & 3) == 3) pt = V2{X, Y};
        const float d = reference_distance(p, pt), e = renderer_distance(p, pt, large);
        // relative above distances of 1 (large coordinates)
        const float diff = std::fabs(d - e) / std::fmax(1.f, d);
        *worst = std::fmax(*worst, diff);
        far += !(diff <= 1e-3f);
        flips += (d < r) != (e < r);
    }
    out[0] = n;
    out[1] = large;
    out[2] = far;
    out[3] = flips;
}
}
