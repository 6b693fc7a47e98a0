// dvg_shade.h -- paints, fragment compositing and boundary sampling on the device.
//
//   sample_paint / d_sample_paint   diffvg.cpp:276-504
//   compositing and its adjoint     diffvg.cpp:525-707 (fragments composited in
//                                   increasing group id, stroke before fill of a group)
//   prefiltered compositing         diffvg.cpp:835-1113
//   sample_boundary                 sample_boundary.h:20-453
//   accumulate_boundary_gradient    diffvg.cpp:89-274
//   gather_d_color                  diffvg.cpp:777-815
// Candidates arrive in increasing group id, so the forward composites each fragment as
// soon as it is found (no fragment list, no sort); the adjoint keeps a per-lane list of
// the fragments and the running accumulation for the reverse sweep.
#pragma once

#include "dvg_query.h"
#include "dvg_wave.h"

namespace dvg {

DVG_DEV V4 stop_color(const float *C, int i) { return V4{C[4 * i], C[4 * i + 1], C[4 * i + 2], C[4 * i + 3]}; }

DVG_DEV V4 sample_paint(const DevScene &S, int type, int off, int ns, V2 pt) {
    const float *c = S.color + off;
    if (type == 0) return V4{c[0], c[1], c[2], c[3]};
    const float *offsets = c + 4;
    const float *colors = c + 4 + ns;
    float t;
    if (type == 1) {
        V2 beg{c[0], c[1]}, end{c[2], c[3]};
        t = dot(pt - beg, end - beg) / fmax_r(dot(end - beg, end - beg), 1e-3f);
    } else {
        V2 center{c[0], c[1]}, radius{c[2], c[3]};
        t = len(vdivv(pt - center, radius));
    }
    if (t < offsets[0]) return stop_color(colors, 0);
    for (int i = 0; i < ns - 1; i++) {
        float oc = offsets[i], on = offsets[i + 1];
        if (t >= oc && t < on) {
            float tt = (t - oc) / (on - oc);
            return stop_color(colors, i) * (1 - tt) + stop_color(colors, i + 1) * tt;
        }
    }
    return stop_color(colors, ns - 1);
}

// d_sample_color; the radial branch keeps the reference's missing `return`.
DVG_DEV void d_sample_paint(const DevScene &S, int type, int off, int ns, V2 pt, V4 d_color, float *d_translation) {
    float *dc = S.d_color + off;
    if (type == 0) {
        aadd4(dc, d_color);
        return;
    }
    const float *c = S.color + off;
    const float *offsets = c + 4;
    const float *colors = c + 4 + ns;
    float *d_offsets = dc + 4;
    float *d_colors = dc + 4 + ns;
    float t;
    V2 a{c[0], c[1]}, b{c[2], c[3]};
    V2 normalized_offset{0, 0}, offset{0, 0};
    if (type == 1) {
        t = dot(pt - a, b - a) / fmax_r(dot(b - a, b - a), 1e-3f);
    } else {
        offset = pt - a;
        normalized_offset = vdivv(offset, b);
        t = len(normalized_offset);
    }
    if (t < offsets[0]) {
        aadd4(d_colors, d_color);
        return;
    }
    for (int i = 0; i < ns - 1; i++) {
        float oc = offsets[i], on = offsets[i + 1];
        if (t >= oc && t < on) {
            V4 cc = stop_color(colors, i), cn = stop_color(colors, i + 1);
            float tt = (t - oc) / (on - oc);
            float d_tt = vsum(d_color * (cn - cc));
            float d_on = -d_tt * tt / (on - oc);
            float d_oc = d_tt * ((tt - 1.f) / (on - oc));
            float d_t = d_tt / (on - oc);
            aadd4(d_colors + 4 * i, d_color * (1 - tt));
            aadd4(d_colors + 4 * (i + 1), d_color * tt);
            aadd(d_offsets + i, d_oc);
            aadd(d_offsets + i + 1, d_on);
            if (type == 1) {
                float l = fmax_r(dot(b - a, b - a), 1e-3f);
                V2 d_beg = vdiv(d_t * (-(pt - a) - (b - a)), l);
                V2 d_end = vdiv(d_t * (pt - a), l);
                float d_l = -d_t * t / l;
                if (dot(b - a, b - a) > 1e-3f) {
                    d_beg += 2 * d_l * (a - b);
                    d_end += 2 * d_l * (b - a);
                }
                aadd2(dc, d_beg);
                aadd2(dc + 2, d_end);
                if (d_translation) aadd2(d_translation, d_beg + d_end);
                return;
            }
            V2 d_no = d_length(normalized_offset, d_t);
            V2 d_offset = vdivv(d_no, b);
            V2 d_radius = vdivv((-d_no) * offset, b * b);
            V2 d_center = -d_offset;
            aadd2(dc, d_center);
            aadd2(dc + 2, d_radius);
            if (d_translation) aadd2(d_translation, d_center);
        }
    }
    aadd4(d_colors + 4 * (ns - 1), d_color);
}

// Running "over" compositor (diffvg.cpp:616-648) with the EdgeQuery bookkeeping
// (diffvg.cpp:624-632): `trav_hit` collects hits raised inside the coverage tests, and
// the per-fragment rules are folded so that the result equals the reference's
// sequential update over the sorted fragment list.
struct Compositor {
    V3 color;
    float alpha;
    int nf;
    bool seen_target, opaque_after_target, any_opaque;
    DVG_DEV void init(bool has_bg, V4 bg) {
        color = has_bg ? V3{bg.x, bg.y, bg.z} : V3{0, 0, 0};
        alpha = has_bg ? bg.w : 0.f;
        nf = 0;
        seen_target = opaque_after_target = any_opaque = false;
    }
    DVG_DEV void add(V4 c, int g, int target_group) {
        if (c.w >= 1.f) {
            any_opaque = true;
            if (seen_target) opaque_after_target = true;
        }
        if (g == target_group) {
            seen_target = true;
            opaque_after_target = false;
        }
        color = color * (1 - c.w) + c.w * V3{c.x, c.y, c.z};
        alpha = alpha * (1 - c.w) + c.w;
        nf++;
    }
    DVG_DEV bool edge_hit(bool trav_hit) const { return seen_target ? !opaque_after_target : (trav_hit && !any_opaque); }
    DVG_DEV V4 result(bool has_bg, V4 bg) const {
        if (nf == 0) return has_bg ? bg : V4{0, 0, 0, 0};
        V3 c = color;
        if (alpha > 1e-6f) c = vdiv(c, alpha);
        return V4{c.x, c.y, c.z, alpha};
    }
};

// Fragment record of the adjoint sweep; the sweep evaluates the fragment's own paint again
// (the records of 64 samples live in scratch memory, which a wave writes and reads whole).
struct FragRec {
    V3 prev_color;
    float prev_alpha;
    int gid;  // group * 2 + is_stroke
};
DVG_DEV V4 frag_paint(const DevScene &S, int gid, V2 pt) {
    const int g = gid >> 1;
    return (gid & 1) ? sample_paint(S, S.stroke_type[g], S.stroke_off[g], S.stroke_ns[g], pt)
                     : sample_paint(S, S.fill_type[g], S.fill_off[g], S.fill_ns[g], pt);
}
constexpr int kMaxFrags = 256;  // the reference's limit (diffvg.cpp:542)

// Reverse compositing sweep (diffvg.cpp:654-705).  Returns the adjoint that reaches the
// background colour.
DVG_DEV V4 composite_adjoint(const DevScene &S, const FragRec *frags, int nf, V3 final_color, float final_alpha,
                             V4 d_color, V2 pt, float *d_translation) {
    V3 d_final_color{d_color.x, d_color.y, d_color.z};
    V3 d_curr_color = d_final_color;
    float d_curr_alpha = d_color.w;
    if (final_alpha > 1e-6f) {
        d_curr_color = vdiv(d_final_color, final_alpha);
        d_curr_alpha -= vsum(d_final_color * final_color) / final_alpha;
    }
    for (int i = nf - 1; i >= 0; i--) {
        const FragRec &f = frags[i];
        const V4 c = frag_paint(S, f.gid, pt);
        float d_prev_alpha = d_curr_alpha * (1.f - c.w);
        float d_alpha_i = d_curr_alpha * (1.f - f.prev_alpha);
        d_alpha_i += vsum(d_curr_color * (V3{c.x, c.y, c.z} - f.prev_color));
        V3 d_prev_color = d_curr_color * (1 - c.w);
        V3 d_color_i = d_curr_color * c.w;
        int g = f.gid >> 1;
        V4 dci{d_color_i.x, d_color_i.y, d_color_i.z, d_alpha_i};
        if (f.gid & 1)
            d_sample_paint(S, S.stroke_type[g], S.stroke_off[g], S.stroke_ns[g], pt, dci, d_translation);
        else
            d_sample_paint(S, S.fill_type[g], S.fill_off[g], S.fill_ns[g], pt, dci, d_translation);
        d_curr_color = d_prev_color;
        d_curr_alpha = d_prev_alpha;
    }
    return V4{d_curr_color.x, d_curr_color.y, d_curr_color.z, d_curr_alpha};
}

// Prefiltered fragment record (diffvg.cpp:514-523)
struct PFragRec {
    V3 color;
    float alpha;
    V3 prev_color;
    float prev_alpha;
    int gid;
    int shape_id;
    float distance;
    V2 closest;
    PathInfo info;
    int within;
};
constexpr int kMaxPFrags = 64;  // diffvg.cpp:847

DVG_DEV V4 composite_adjoint_prefiltered(const DevScene &S, const PFragRec *frags, int nf, V3 final_color,
                                         float final_alpha, V4 d_color, V2 pt, float *d_translation) {
    V3 d_final_color{d_color.x, d_color.y, d_color.z};
    V3 d_curr_color = d_final_color;
    float d_curr_alpha = d_color.w;
    if (final_alpha > 1e-6f) {
        d_curr_color = vdiv(d_final_color, final_alpha);
        d_curr_alpha -= vsum(d_final_color * final_color) / final_alpha;
    }
    for (int i = nf - 1; i >= 0; i--) {
        const PFragRec &f = frags[i];
        float d_prev_alpha = d_curr_alpha * (1.f - f.alpha);
        float d_alpha_i = d_curr_alpha * (1.f - f.prev_alpha);
        d_alpha_i += vsum(d_curr_color * (f.color - f.prev_color));
        V3 d_prev_color = d_curr_color * (1 - f.alpha);
        V3 d_color_i = d_curr_color * f.alpha;
        int g = f.gid >> 1;
        int s = f.shape_id;
        float d = f.distance;
        if (f.gid & 1) {
            float sw = S.stroke_width[s];
            float ad = (float)fabs((double)d);
            float apw = ad + sw, amw = ad - sw;
            float w = smoothstep(apw) - smoothstep(amw);
            if (w != 0) {
                float d_w = w > 0 ? (f.alpha / w) * d_alpha_i : 0.f;
                d_alpha_i *= w;
                d_sample_paint(S, S.stroke_type[g], S.stroke_off[g], S.stroke_ns[g], pt,
                               V4{d_color_i.x, d_color_i.y, d_color_i.z, d_alpha_i}, d_translation);
                float d_apw = d_smoothstep(apw, d_w);
                float d_amw = -d_smoothstep(amw, d_w);
                float d_d = d_apw + d_amw;
                if (d < 0) d_d = -d_d;
                float d_sw = d_apw - d_amw;
                if (fabs((double)d_d) > 1e-10f) d_compute_distance(S, g, s, pt, f.closest, f.info, d_d, d_translation);
                aadd(S.d_stroke_width + s, d_sw);
            }
        } else {
            float w = smoothstep(d);
            if (w != 0) {
                float d_w = w > 0 ? (f.alpha / w) * d_alpha_i : 0.f;
                d_alpha_i *= w;
                d_sample_paint(S, S.fill_type[g], S.fill_off[g], S.fill_ns[g], pt,
                               V4{d_color_i.x, d_color_i.y, d_color_i.z, d_alpha_i}, d_translation);
                float d_d = d_smoothstep(d, d_w);
                if (d < 0) d_d = -d_d;
                if (fabs((double)d_d) > 1e-10f && f.within)
                    d_compute_distance(S, g, s, pt, f.closest, f.info, d_d, d_translation);
            }
        }
        d_curr_color = d_prev_color;
        d_curr_alpha = d_prev_alpha;
    }
    return V4{d_curr_color.x, d_curr_color.y, d_curr_color.z, d_curr_alpha};
}

// gather_d_color (diffvg.cpp:777-815)
DVG_DEV V4 gather_d_color(int ftype, float radius, const float *d_img, const float *w_img, int W, int H, V2 pt) {
    int x = (int)pt.x, y = (int)pt.y;
    int ri = (int)ceil((double)radius);
    V4 d_color{0, 0, 0, 0};
    for (int dy = -ri; dy <= ri; dy++) {
        for (int dx = -ri; dx <= ri; dx++) {
            int xx = x + dx, yy = y + dy;
            if (xx >= 0 && xx < W && yy >= 0 && yy < H) {
                float xc = xx + 0.5f, yc = yy + 0.5f;
                float fw = filter_weight(ftype, radius, xc - pt.x, yc - pt.y);
                float ws = w_img[yy * W + xx];
                if (ws > 0) {
                    float4 d = reinterpret_cast<const float4 *>(d_img)[yy * W + xx];
                    d_color += (fw / ws) * V4{d.x, d.y, d.z, d.w};
                }
            }
        }
    }
    return d_color;
}

// gather_d_color at a sample's point and the filter-radius adjoint of the sample's splat
// (diffvg.cpp:1250-1268), which visit the same taps: one pass loads each and evaluates its
// filter once (the double-precision exponential of a Gaussian is what it costs).  The gather
// is centred on the pixel the point lies in, the splat on the sample's own pixel (x, y); they
// differ where the jittered position rounds up to the next pixel.  k_color_bwd of 300 paths at
// 512x512, Gaussian of radius 1.5: 337 -> 268 us, prefiltered 743 -> 664.
DVG_DEV V4 gather_and_splat_adjoint(int ftype, float radius, const float *d_img, const float *w_img, int W, int H,
                                    V2 pt, int x, int y, V4 color, float &d_radius) {
    const int ri = (int)ceil((double)radius);
    const double r5 = ftype == kTent ? pow((double)radius, 5.0) : 1.0;
    V4 d_color{0, 0, 0, 0};
    const bool same = (int)pt.x == x && (int)pt.y == y;
    for (int pass = 0; pass < (same ? 1 : 2); pass++) {
        const bool gather = pass == 0, splat = same || pass == 1;
        const int cx = gather ? (int)pt.x : x, cy = gather ? (int)pt.y : y;
        for (int dy = -ri; dy <= ri; dy++)
            for (int dx = -ri; dx <= ri; dx++) {
                const int xx = cx + dx, yy = cy + dy;
                if (xx < 0 || xx >= W || yy < 0 || yy >= H) continue;
                const float ws = w_img[yy * W + xx];
                if (!(ws > 0)) continue;
                const float fx = xx + 0.5f - pt.x, fy = yy + 0.5f - pt.y;
                const FilterTap tap = filter_tap(ftype, radius, fx, fy);
                const float4 d4 = reinterpret_cast<const float4 *>(d_img)[yy * W + xx];
                const V4 d{d4.x, d4.y, d4.z, d4.w};
                if (gather) d_color += (tap.w / ws) * d;
                if (splat) {
                    const float dpc = dot(d, color);
                    const float d_weight = (dpc * ws - tap.w * dpc * (ws - tap.w)) / (ws * ws);
                    d_radius += filter_tap_adjoint(tap, ftype, radius, r5, fx, fy, d_weight);
                }
            }
    }
    return d_color;
}

// ---------------------------------------------------------------- boundary sampling
struct BoundaryData {
    int base_point_id, point_id;
    float t;
    int is_stroke;
};

// Edge sample record, 64 bytes (BoundarySample, diffvg.cpp:1314-1323)
struct alignas(16) EdgeSample {
    float px, py;          // normalised canvas position
    float lx, ly;          // local boundary point
    float nx, ny;          // canvas normal
    int group, shape;      // shape < 0: invalid sample
    float t;
    float pdf;
    BoundaryData data;
};

DVG_DEV int cdf_sample(const float *cdf, int n, float u, float *updated_u) {
    int lb = 0;
    int len_ = n - 1 - lb;
    while (len_ > 0) {
        int half = len_ / 2;
        int mid = lb + half;
        if (u < cdf[mid]) {
            len_ = half;
        } else {
            lb = mid + 1;
            len_ = len_ - half - 1;
        }
    }
    lb = lb < 0 ? 0 : (lb > n - 1 ? n - 1 : lb);
    if (updated_u) {
        if (lb > 0)
            *updated_u = (u - cdf[lb - 1]) / (cdf[lb] - cdf[lb - 1]);
        else
            *updated_u = u / cdf[lb];
    }
    return lb;
}

DVG_DEV V2 perturb(V2 ret, float dir, float r, V2 &normal) {
    if (dir != 0.f) {
        ret += dir * r * normal;
        if (dir < 0) normal = -normal;
    }
    return ret;
}

DVG_DEV V2 sample_boundary(const DevScene &S, int g, int s, float t, V2 &normal, float &pdf, BoundaryData &data) {
    pdf = 1;
    bool stroke_perturb = false;
    bool has_fill = S.fill_type[g] >= 0, has_stroke = S.stroke_type[g] >= 0;
    if (has_fill && has_stroke) {
        if (t < 0.5f) {
            t = 2 * t;
        } else {
            stroke_perturb = true;
            t = 2 * (t - 0.5f);
        }
        pdf = 0.5f;
    } else if (has_stroke) {
        stroke_perturb = true;
    }
    data.is_stroke = stroke_perturb;
    float dir = 0.f;
    if (stroke_perturb) {
        if (t < 0.5f) {
            dir = -1.f;
            t = 2 * t;
        } else {
            dir = 1.f;
            t = 2 * (t - 0.5f);
        }
        pdf *= 0.5f;
    }
    float sr = S.stroke_width[s];
    int type = S.shape_type[s];
    const float tp = 2 * (float)kPi;
    if (type != 2) {
        const float *P = S.params + S.param_off[s];
        if (type == 0) {
            V2 offset{(float)((double)P[0] * cos((double)(tp * t))), (float)((double)P[0] * sin((double)(tp * t)))};
            normal = normalize(offset);
            pdf /= (tp * P[0]);
            return perturb(V2{P[1], P[2]} + offset, dir, sr, normal);
        } else if (type == 1) {
            V2 offset{(float)((double)P[0] * cos((double)(tp * t))), (float)((double)P[1] * sin((double)(tp * t)))};
            double dxdt = (double)-P[0] * sin((double)(tp * t)) * 2 * (double)(float)kPi;
            double dydt = (double)P[1] * cos((double)(tp * t)) * 2 * (double)(float)kPi;
            normal = normalize(V2{(float)dydt, (float)-dxdt});
            pdf = (float)((double)pdf / sqrt(dxdt * dxdt + dydt * dydt));
            return perturb(V2{P[2], P[3]} + offset, dir, sr, normal);
        }
        float w = P[2] - P[0], h = P[3] - P[1];
        pdf /= (2 * (w + h));
        if (t <= w / (w + h)) {
            t *= (w + h) / w;
            if (t < 0.5f) {
                normal = V2{0, -1};
                return perturb(V2{P[0], P[1]} + 2 * t * V2{P[2] - P[0], 0.f}, dir, sr, normal);
            }
            normal = V2{0, 1};
            return perturb(V2{P[0], P[3]} + 2 * (t - 0.5f) * V2{P[2] - P[0], 0.f}, dir, sr, normal);
        }
        t = (t - w / (w + h)) * (w + h) / h;
        if (t < 0.5f) {
            normal = V2{-1, 0};
            return perturb(V2{P[0], P[1]} + 2 * t * V2{0.f, P[3] - P[1]}, dir, sr, normal);
        }
        normal = V2{1, 0};
        return perturb(V2{P[2], P[1]} + 2 * (t - 0.5f) * V2{0.f, P[3] - P[1]}, dir, sr, normal);
    }
    bool thick = S.has_thick[s] != 0;
    int np = S.npt[s], po = S.pt_off[s];
    int sb = S.seg_begin[s], nb = S.nsegs[s];
    if (dir != 0.f && !S.closed[s]) {
        float cap_length = thick ? (float)kPi * (S.thickness[po] + S.thickness[po + np - 1]) : 2 * (float)kPi * sr;
        float cap_prob = cap_length / (cap_length + S.shape_length[s]);
        if (t < cap_prob) {
            t = t / cap_prob;
            pdf *= cap_prob;
            float r0 = thick ? S.thickness[po] : sr;
            float r1 = thick ? S.thickness[po + np - 1] : sr;
            float rr = dir < 0 ? r0 : r1;
            V2 p0 = dir < 0 ? ld_pt(S, po) : ld_pt(S, po + np - 1);
            V2 offset{(float)((double)rr * cos((double)(tp * t))), (float)((double)rr * sin((double)(tp * t)))};
            normal = normalize(offset);
            pdf /= (tp * rr);
            if (dir < 0) {
                data.base_point_id = 0;
                data.point_id = 0;
                data.t = 0;
            } else {
                data.base_point_id = nb - 1;
                data.point_id = np - 2 - S.seg_kind[sb + nb - 1];
                data.t = 1;
            }
            return p0 + offset;
        }
        t = (t - cap_prob) / (1 - cap_prob);
        pdf *= (1 - cap_prob);
    }
    int sample_id = cdf_sample(S.seg_cdf + sb, nb, t, &t);
    int seg = sb + sample_id;
    V2 p[4];
    int4 idx;
    int k = seg_load(S, seg, p, idx);
    data.base_point_id = sample_id;
    data.point_id = S.seg_pid[seg];
    data.t = t;
    if (t < -1e-3f || t > 1 + 1e-3f) {
        pdf = 0;
        return V2{0, 0};
    }
    V2 tangent, ret;
    float rr;
    if (k == 0) {
        tangent = p[1] - p[0];
        ret = p[0] + t * (p[1] - p[0]);
        float r0 = thick ? S.thickness[idx.x] : sr, r1 = thick ? S.thickness[idx.y] : sr;
        rr = r0 + t * (r1 - r0);
    } else if (k == 1) {
        tangent = 2 * (1 - t) * (p[1] - p[0]) + 2 * t * (p[2] - p[1]);
        ret = qeval(p[0], p[1], p[2], t);
        float r0 = thick ? S.thickness[idx.x] : sr, r1 = thick ? S.thickness[idx.y] : sr,
              r2 = thick ? S.thickness[idx.z] : sr;
        float tt = 1 - t;
        rr = (tt * tt) * r0 + (2 * tt * t) * r1 + (t * t) * r2;
    } else {
        float omt = 1 - t;
        tangent = 3 * (omt * omt) * (p[1] - p[0]) + 6 * (1 - t) * t * (p[2] - p[1]) + 3 * t * t * (p[3] - p[2]);
        ret = ceval(p[0], p[1], p[2], p[3], t);
        float r0 = thick ? S.thickness[idx.x] : sr, r1 = thick ? S.thickness[idx.y] : sr,
              r2 = thick ? S.thickness[idx.z] : sr, r3 = thick ? S.thickness[idx.w] : sr;
        float tt = 1 - t;
        rr = (tt * tt * tt) * r0 + (3 * tt * tt * t) * r1 + (3 * tt * t * t) * r2 + (t * t * t) * r3;
    }
    float tan_len = len(tangent);
    if (tan_len == 0) {
        pdf = 0;
        return V2{0, 0};
    }
    normal = vdiv(V2{-tangent.y, tangent.x}, tan_len);
    pdf *= S.seg_pmf[seg] / tan_len;
    if (dir != 0.f) {
        ret += dir * rr * normal;
        if (dir < 0) normal = -normal;
    }
    return ret;
}

// sample_boundary_kernel body (diffvg.cpp:1325-1386): fills `es`, returns validity.
DVG_DEV bool make_edge_sample(const DevScene &S, int idx, uint64_t seed, EdgeSample &es) {
    es.shape = -1;
    Pcg rng = pcg_init(idx, seed);
    float u = pcg_float(rng);
    int sample_id = cdf_sample(S.shapes_cdf, S.num_total_shapes, u, nullptr);
    int s = S.sample_shape_id[sample_id];
    int g = S.sample_group_id[sample_id];
    float shape_pmf = S.shapes_pmf[s];  // indexed by shape id, as the reference does
    if (shape_pmf <= 0) return false;
    float t = pcg_float(rng);
    V2 normal{0, 0};
    float pdf = 0.f;
    BoundaryData bd{0, 0, 0.f, 0};
    V2 lp = sample_boundary(S, g, s, t, normal, pdf, bd);
    if (pdf <= 0) return false;
    M3 s2c = m3_load(S.s2c + 9 * g);
    M3 c2s = m3_load(S.c2s + 9 * g);
    V2 bpt = xform_pt(s2c, lp);
    normal = xform_normal(c2s, normal);
    bpt.x /= S.cw;
    bpt.y /= S.ch;
    es.px = bpt.x;
    es.py = bpt.y;
    es.lx = lp.x;
    es.ly = lp.y;
    es.nx = normal.x;
    es.ny = normal.y;
    es.group = g;
    es.shape = s;
    es.t = t;
    es.pdf = shape_pmf * pdf;
    es.data = bd;
    return true;
}

// accumulate_boundary_gradient (diffvg.cpp:89-274)
DVG_DEV void accumulate_boundary_gradient(const DevScene &S, int g, int s, float contrib, float t, V2 normal,
                                          const BoundaryData &bd, V2 local_pt) {
    int type = S.shape_type[s];
    if (bd.is_stroke) {
        if (type == 2 && S.has_thick[s]) {
            int seg = S.seg_begin[s] + bd.base_point_id;
            int4 idx = S.seg_idx[seg];
            int k = S.seg_kind[seg];
            float tt = bd.t;
            if (k == 0) {
                aadd(S.d_thickness + idx.x, (1 - tt) * contrib);
                aadd(S.d_thickness + idx.y, (tt)*contrib);
            } else if (k == 1) {
                aadd(S.d_thickness + idx.x, ((1 - tt) * (1 - tt)) * contrib);
                aadd(S.d_thickness + idx.y, (2 * (1 - tt) * tt) * contrib);
                aadd(S.d_thickness + idx.z, (tt * tt) * contrib);
            } else {
                float o = 1 - tt;
                aadd(S.d_thickness + idx.x, (o * o * o) * contrib);
                aadd(S.d_thickness + idx.y, 3 * (o * o) * tt * contrib);
                aadd(S.d_thickness + idx.z, 3 * (1 - tt) * tt * tt * contrib);
                aadd(S.d_thickness + idx.w, tt * tt * tt * contrib);
            }
        } else {
            aadd(S.d_stroke_width + s, contrib);
        }
    }
    if (type == 0) {
        float *dp = S.d_params + S.param_off[s];
        aadd2(dp + 1, normal * contrib);
        aadd(dp, contrib);
    } else if (type == 1) {
        float *dp = S.d_params + S.param_off[s];
        const float tp = 2 * (float)kPi;
        aadd2(dp + 2, normal * contrib);
        aadd(dp + 0, (float)(cos((double)(tp * t)) * normal.x * contrib));
        aadd(dp + 1, (float)(sin((double)(tp * t)) * normal.y * contrib));
    } else if (type == 2) {
        int seg = S.seg_begin[s] + bd.base_point_id;
        int4 idx = S.seg_idx[seg];
        int k = S.seg_kind[seg];
        float tt = bd.t;
        float w[4];
        int ii[4] = {idx.x, idx.y, idx.z, idx.w};
        if (k == 0) {
            w[0] = 1 - tt;
            w[1] = tt;
        } else if (k == 1) {
            w[0] = (1 - tt) * (1 - tt);
            w[1] = 2 * (1 - tt) * tt;
            w[2] = tt * tt;
        } else {
            float o = 1 - tt;
            w[0] = o * o * o;
            w[1] = 3 * (o * o) * tt;
            w[2] = 3 * (1 - tt) * tt * tt;
            w[3] = tt * tt * tt;
        }
        for (int j = 0; j <= k + 1; j++) {
            aadd(S.d_points + 2 * ii[j] + 0, w[j] * normal.x * contrib);
            aadd(S.d_points + 2 * ii[j] + 1, w[j] * normal.y * contrib);
        }
    } else {
        float *dp = S.d_params + S.param_off[s];
        if (normal == V2{-1, 0})
            aadd(dp + 0, -contrib);
        else if (normal == V2{1, 0})
            aadd(dp + 2, contrib);
        else if (normal == V2{0, -1})
            aadd(dp + 1, -contrib);
        else if (normal == V2{0, 1})
            aadd(dp + 3, contrib);
    }
    M3 s2c = m3_load(S.s2c + 9 * g);
    M3 d_s2c;
#pragma unroll
    for (int i = 0; i < 9; i++) d_s2c.m[i] = 0.f;
    V2 d_local{0, 0};
    d_xform_pt(s2c, local_pt, normal * contrib, d_s2c, d_local);
    float *dx = S.d_xform + 9 * g;
#pragma unroll
    for (int i = 0; i < 9; i++) aadd(dx + i, d_s2c.m[i]);
}

// Offset of the gradient copy this workgroup adds to (DevScene::rep_mask).
DVG_DEV int grad_copy(const DevScene &S) { return (int)(blockIdx.x & (unsigned)S.rep_mask) * S.rep_stride; }

// ---- wave-combined gradient scatter for boundary samples ----
// Device-scope float atomics to ordinary device memory are resolved past the XCD's L2,
// so the ~20 atomics per boundary sample dominate the edge kernel's memory traffic.  A
// wave's boundary samples come from one pixel tile and mostly share a few shapes and
// segments: lanes with equal keys add their values in registers first and one lane
// issues the atomics.  Must be called by every lane of the wave (inactive lanes pass
// active = false).
template <int N>
DVG_DEV void wave_combine_add(bool active, int key, const float (&v)[N], float *dst_of_key_leader,
                              int n_used = N) {
    const int lane = threadIdx.x & 63;
    uint64_t pending = __ballot(active);
    while (pending) {
        const int leader = __ffsll((unsigned long long)pending) - 1;
        const int lk = __shfl(key, leader, 64);
        const bool mine = active && key == lk && ((pending >> lane) & 1ull);
        const uint64_t m = __ballot(mine);
        float sum[N];
#pragma unroll
        for (int i = 0; i < N; i++) {
            float x = mine ? v[i] : 0.f;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
            sum[i] = x;
        }
        // the destination of this key, as the leader computed it; the N contiguous sums go
        // out as one atomic instruction of N lanes
        const unsigned long long addr =
            ((unsigned long long)(unsigned)__shfl((int)((unsigned long long)dst_of_key_leader >> 32), leader, 64)
             << 32) |
            (unsigned)__shfl((int)((unsigned long long)dst_of_key_leader & 0xffffffffull), leader, 64);
        const int nu = N == 1 ? 1 : __shfl(n_used, leader, 64);
        float mine_sum = sum[0];
#pragma unroll
        for (int i = 1; i < N; i++) mine_sum = lane == i ? sum[i] : mine_sum;
        if (lane < nu) aadd((float *)addr + lane, mine_sum);
        pending &= ~m;
    }
}

// accumulate_boundary_gradient (diffvg.cpp:89-274) for a whole wave: the same values as
// the per-sample version, with the stroke-width, path-point and transform adjoints of
// lanes that share a shape, segment or group added together before the atomics.
DVG_DEV void accumulate_boundary_gradient_wave(const DevScene &S, bool active, int g, int s, float contrib, float t,
                                               V2 normal, const BoundaryData &bd, V2 local_pt, bool prim_direct) {
    int type = active ? S.shape_type[s] : -1;
    // strokes: per-point thickness goes direct (rare); stroke width combined by shape
    bool sw_active = active && bd.is_stroke && !(type == 2 && S.has_thick[s]);
    if (active && bd.is_stroke && type == 2 && S.has_thick[s]) {
        int seg = S.seg_begin[s] + bd.base_point_id;
        int4 idx = S.seg_idx[seg];
        int k = S.seg_kind[seg];
        float tt = bd.t;
        if (k == 0) {
            aadd(S.d_thickness + idx.x, (1 - tt) * contrib);
            aadd(S.d_thickness + idx.y, (tt)*contrib);
        } else if (k == 1) {
            aadd(S.d_thickness + idx.x, ((1 - tt) * (1 - tt)) * contrib);
            aadd(S.d_thickness + idx.y, (2 * (1 - tt) * tt) * contrib);
            aadd(S.d_thickness + idx.z, (tt * tt) * contrib);
        } else {
            float o = 1 - tt;
            aadd(S.d_thickness + idx.x, (o * o * o) * contrib);
            aadd(S.d_thickness + idx.y, 3 * (o * o) * tt * contrib);
            aadd(S.d_thickness + idx.z, 3 * (1 - tt) * tt * tt * contrib);
            aadd(S.d_thickness + idx.w, tt * tt * tt * contrib);
        }
    }
    {
        float v[1] = {contrib};
        wave_combine_add<1>(sw_active, s, v, S.d_stroke_width + grad_copy(S) + (sw_active ? s : 0));
    }
    // shape parameters of circles, ellipses and rects: combined by shape, or (prim_direct,
    // see kPrimDirect) added by every lane
    if (prim_direct) {
        if (active && type == 0) {
            float *dp = S.d_params + S.param_off[s];
            aadd2(dp + 1, normal * contrib);
            aadd(dp, contrib);
        } else if (active && type == 1) {
            float *dp = S.d_params + S.param_off[s];
            const float tp = 2 * (float)kPi;
            aadd2(dp + 2, normal * contrib);
            aadd(dp + 0, (float)(cos((double)(tp * t)) * normal.x * contrib));
            aadd(dp + 1, (float)(sin((double)(tp * t)) * normal.y * contrib));
        } else if (active && type == 3) {
            float *dp = S.d_params + S.param_off[s];
            if (normal == V2{-1, 0})
                aadd(dp + 0, -contrib);
            else if (normal == V2{1, 0})
                aadd(dp + 2, contrib);
            else if (normal == V2{0, -1})
                aadd(dp + 1, -contrib);
            else if (normal == V2{0, 1})
                aadd(dp + 3, contrib);
        }
    } else {
        float v[4] = {0.f, 0.f, 0.f, 0.f};
        const bool on = active && type != 2;
        int n = 4;
        if (on && type == 0) {
            v[0] = contrib;
            v[1] = normal.x * contrib;
            v[2] = normal.y * contrib;
            n = 3;
        } else if (on && type == 1) {
            const float tp = 2 * (float)kPi;
            v[0] = (float)(cos((double)(tp * t)) * normal.x * contrib);
            v[1] = (float)(sin((double)(tp * t)) * normal.y * contrib);
            v[2] = normal.x * contrib;
            v[3] = normal.y * contrib;
        } else if (on) {
            if (normal == V2{-1, 0})
                v[0] = -contrib;
            else if (normal == V2{1, 0})
                v[2] = contrib;
            else if (normal == V2{0, -1})
                v[1] = -contrib;
            else if (normal == V2{0, 1})
                v[3] = contrib;
        }
        wave_combine_add<4>(on, s, v, S.d_params + grad_copy(S) + (on ? S.param_off[s] : 0), n);
    }
    // path control points, combined by segment.  A segment's points are not contiguous
    // (the last point of a closed path's last segment wraps to its first), so each of the
    // up to four points is combined and added separately, keyed by segment.
    {
        bool pa = active && type == 2;
        int seg = pa ? S.seg_begin[s] + bd.base_point_id : 0;
        int4 idx = pa ? S.seg_idx[seg] : make_int4(0, 0, 0, 0);
        int k = pa ? S.seg_kind[seg] : 0;
        float tt = bd.t;
        float w[4] = {0.f, 0.f, 0.f, 0.f};
        if (k == 0) {
            w[0] = 1 - tt;
            w[1] = tt;
        } else if (k == 1) {
            w[0] = (1 - tt) * (1 - tt);
            w[1] = 2 * (1 - tt) * tt;
            w[2] = tt * tt;
        } else {
            float o = 1 - tt;
            w[0] = o * o * o;
            w[1] = 3 * (o * o) * tt;
            w[2] = 3 * (1 - tt) * tt * tt;
            w[3] = tt * tt * tt;
        }
        int ii[4] = {idx.x, idx.y, idx.z, idx.w};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            bool on = pa && j <= k + 1;
            float v[2] = {w[j] * normal.x * contrib, w[j] * normal.y * contrib};
            wave_combine_add<2>(on, seg, v, S.d_points + grad_copy(S) + (on ? 2 * ii[j] : 0));
        }
    }
    // shape_to_canvas adjoint, combined by group
    {
        float m9[9];
        if (active) {
            M3 s2c = m3_load(S.s2c + 9 * g);
            M3 d_s2c;
#pragma unroll
            for (int i = 0; i < 9; i++) d_s2c.m[i] = 0.f;
            V2 d_local{0, 0};
            d_xform_pt(s2c, local_pt, normal * contrib, d_s2c, d_local);
#pragma unroll
            for (int i = 0; i < 9; i++) m9[i] = d_s2c.m[i];
        } else {
#pragma unroll
            for (int i = 0; i < 9; i++) m9[i] = 0.f;
        }
        wave_combine_add<9>(active, g, m9, S.d_xform + grad_copy(S) + (active ? 9 * g : 0));
    }
}

// accumulate_boundary_gradient_wave with the sums of a wave's samples gathered in LDS: lanes
// of one (group, shape, segment) take a row of a table, each value is one LDS atomic
// instruction whatever the number of rows, and the rows then leave as atomics 64 at a time.
// The register form reduces 18 values across the wave once per distinct row, ~20 rows of 64
// samples: k_edge of 2048 strokes at 512x512, 4 samples, 1.48 -> 1.30 ms; 300 paths 0.88 -> 0.79.
constexpr int kScatterVals = 18;  // stroke width, up to 4 points or parameters (8), transform (9)
struct ScatterLds {
    float row[64][kScatterVals];
    int group[64], shape[64], seg[64];
};
DVG_DEV void accumulate_boundary_gradient_lds(const DevScene &S, ScatterLds &L, bool active, int g, int s,
                                              float contrib, float t, V2 normal, const BoundaryData &bd, V2 local_pt,
                                              bool prim_direct) {
    const int lane = threadIdx.x & 63;
    const int type = active ? S.shape_type[s] : -1;
    const bool path = type == 2;
    const int seg = path ? S.seg_begin[s] + bd.base_point_id : -1;
    // rows
    int mine = -1, head = -1, rows = 0;  // head: the first row of the lane's (group, shape)
    for (uint64_t pending = __ballot(active); pending;) {
        const int leader = __ffsll((unsigned long long)pending) - 1;
        const int lg = __builtin_amdgcn_readlane(g, leader), ls = __builtin_amdgcn_readlane(s, leader),
                  lseg = __builtin_amdgcn_readlane(seg, leader);
        const bool shape = active && g == lg && s == ls, same = shape && seg == lseg;
        if (shape && head < 0) head = rows;
        const uint64_t m = __ballot(same);
        if (same) mine = rows;
        pending &= ~m;
        rows++;
    }
    wave_sync();
    for (int i = lane; i < rows * kScatterVals; i += 64) (&L.row[0][0])[i] = 0.f;
    if (active) {  // lanes of one row write the same values
        L.group[mine] = g;
        L.shape[mine] = s;
        L.seg[mine] = seg;
    }
    wave_sync();
    if (active) {
        // width and transform go to the head row: a wave on a path of many segments would
        // send up to 64 atomics to the same nine addresses (1500-segment path: k_edge
        // 0.25 -> 0.22 ms)
        float *row = L.row[mine], *row0 = L.row[head];
        auto add_to = [](float *row, int i, float v) {
            __hip_atomic_fetch_add(row + i, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        };
        auto add = [&](int i, float v) { add_to(row, i, v); };
        if (bd.is_stroke && !(path && S.has_thick[s])) add_to(row0, 0, contrib);
        if (path) {
            const int k = S.seg_kind[seg];
            const float tt = bd.t, o = 1 - tt;
            float w[4] = {0.f, 0.f, 0.f, 0.f};
            if (k == 0) {
                w[0] = 1 - tt;
                w[1] = tt;
            } else if (k == 1) {
                w[0] = (1 - tt) * (1 - tt);
                w[1] = 2 * (1 - tt) * tt;
                w[2] = tt * tt;
            } else {
                w[0] = o * o * o;
                w[1] = 3 * (o * o) * tt;
                w[2] = 3 * (1 - tt) * tt * tt;
                w[3] = tt * tt * tt;
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (j > k + 1) break;
                add(1 + 2 * j, w[j] * normal.x * contrib);
                add(2 + 2 * j, w[j] * normal.y * contrib);
            }
            if (bd.is_stroke && S.has_thick[s]) {  // per-point thickness (rare)
                const int4 idx = S.seg_idx[seg];
                const int ii[4] = {idx.x, idx.y, idx.z, idx.w};
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (j <= k + 1) aadd(S.d_thickness + ii[j], w[j] * contrib);
            }
        } else {
            float v[4] = {0.f, 0.f, 0.f, 0.f};
            int n = 4;
            if (type == 0) {
                v[0] = contrib;
                v[1] = normal.x * contrib;
                v[2] = normal.y * contrib;
                n = 3;
            } else if (type == 1) {
                const float tp = 2 * (float)kPi;
                v[0] = (float)(cos((double)(tp * t)) * normal.x * contrib);
                v[1] = (float)(sin((double)(tp * t)) * normal.y * contrib);
                v[2] = normal.x * contrib;
                v[3] = normal.y * contrib;
            } else if (normal == V2{-1, 0}) {
                v[0] = -contrib;
            } else if (normal == V2{1, 0}) {
                v[2] = contrib;
            } else if (normal == V2{0, -1}) {
                v[1] = -contrib;
            } else if (normal == V2{0, 1}) {
                v[3] = contrib;
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (j >= n) break;
                if (v[j] == 0.f) continue;  // a rectangle's sample moves one side
                if (prim_direct)  // see kPrimDirect
                    aadd(S.d_params + S.param_off[s] + j, v[j]);
                else
                    add(1 + j, v[j]);
            }
        }
        const M3 s2c = m3_load(S.s2c + 9 * g);
        M3 d_s2c;
#pragma unroll
        for (int i = 0; i < 9; i++) d_s2c.m[i] = 0.f;
        V2 d_local{0, 0};
        d_xform_pt(s2c, local_pt, normal * contrib, d_s2c, d_local);
#pragma unroll
        for (int i = 0; i < 9; i++) add_to(row0, 9 + i, d_s2c.m[i]);
    }
    wave_sync();
    const int copy = grad_copy(S);
    for (int i = lane; i < rows * kScatterVals; i += 64) {
        const float v = (&L.row[0][0])[i];
        if (v == 0.f) continue;  // also the values a row does not have
        const int r = i / kScatterVals, c = i - r * kScatterVals, rs = L.shape[r], rseg = L.seg[r];
        float *dst;
        if (c == 0) {
            dst = S.d_stroke_width + rs;
        } else if (c >= 9) {
            dst = S.d_xform + 9 * L.group[r] + (c - 9);
        } else if (rseg >= 0) {
            const int j = (c - 1) >> 1;
            dst = S.d_points + 2 * reinterpret_cast<const int *>(S.seg_idx + rseg)[j] + ((c - 1) & 1);
        } else {
            dst = S.d_params + S.param_off[rs] + (c - 1);
        }
        aadd(dst + copy, v);
    }
}

// d_sample_paint for a whole wave (every lane calls it; lanes without a paint adjoint pass
// on = false): lanes that add to the same stops or the same gradient end points add their
// values together before the atomics.  A drawing's gradient fill covers thousands of samples
// that all add to its few stops.  A stop offset order that lets one value fall into several
// intervals of a radial paint (possible only when the offsets are not sorted) adds the later
// ones per lane.
DVG_DEV void d_sample_paint_wave(const DevScene &S, bool on, int type, int off, int ns, V2 pt, V4 d_color,
                                 float *d_translation) {
    // the colour that receives all of d_color: a constant paint, the first stop before the
    // first offset, the last stop past the last (and, for radial paints, always)
    int full = on ? off : -1;
    const bool grad = on && type != 0;
    if (__any(grad)) {
        float geo[4] = {0.f, 0.f, 0.f, 0.f}, offs[2] = {0.f, 0.f}, cols[8];
#pragma unroll
        for (int k = 0; k < 8; k++) cols[k] = 0.f;
        int at = -1;
        if (grad) {
            const float *c = S.color + off;
            const float *offsets = c + 4;
            const float *colors = c + 4 + ns;
            const V2 a{c[0], c[1]}, b{c[2], c[3]};
            V2 normalized_offset{0, 0}, offset{0, 0};
            float t;
            if (type == 1) {
                t = dot(pt - a, b - a) / fmax_r(dot(b - a, b - a), 1e-3f);
            } else {
                offset = pt - a;
                normalized_offset = vdivv(offset, b);
                t = len(normalized_offset);
            }
            full = off + 4 + ns + 4 * (ns - 1);
            const bool before = t < offsets[0];
            if (before) full = off + 4 + ns;
            for (int i = 0; i < ns - 1 && !before; i++) {
                const float oc = offsets[i], ox = offsets[i + 1];
                if (!(t >= oc && t < ox)) continue;
                const V4 cc = stop_color(colors, i), cn = stop_color(colors, i + 1);
                const float tt = (t - oc) / (ox - oc);
                const float d_tt = vsum(d_color * (cn - cc));
                const float d_ox = -d_tt * tt / (ox - oc);
                const float d_oc = d_tt * ((tt - 1.f) / (ox - oc));
                const float d_t = d_tt / (ox - oc);
                const V4 dc = d_color * (1 - tt), dn = d_color * tt;
                V2 d_a, d_b;
                if (type == 1) {
                    const float l = fmax_r(dot(b - a, b - a), 1e-3f);
                    d_a = vdiv(d_t * (-(pt - a) - (b - a)), l);
                    d_b = vdiv(d_t * (pt - a), l);
                    const float d_l = -d_t * t / l;
                    if (dot(b - a, b - a) > 1e-3f) {
                        d_a += 2 * d_l * (a - b);
                        d_b += 2 * d_l * (b - a);
                    }
                    if (d_translation) aadd2(d_translation, d_a + d_b);
                } else {
                    const V2 d_no = d_length(normalized_offset, d_t);
                    d_a = -vdivv(d_no, b);
                    d_b = vdivv((-d_no) * offset, b * b);
                    if (d_translation) aadd2(d_translation, d_a);
                }
                if (at < 0) {
                    at = i;
                    geo[0] = d_a.x, geo[1] = d_a.y, geo[2] = d_b.x, geo[3] = d_b.y;
                    offs[0] = d_oc, offs[1] = d_ox;
                    cols[0] = dc.x, cols[1] = dc.y, cols[2] = dc.z, cols[3] = dc.w;
                    cols[4] = dn.x, cols[5] = dn.y, cols[6] = dn.z, cols[7] = dn.w;
                } else {
                    float *d = S.d_color + off;
                    aadd2(d, d_a);
                    aadd2(d + 2, d_b);
                    aadd(d + 4 + i, d_oc);
                    aadd(d + 4 + i + 1, d_ox);
                    aadd4(d + 4 + ns + 4 * i, dc);
                    aadd4(d + 4 + ns + 4 * (i + 1), dn);
                }
                if (type == 1) {
                    full = -1;
                    break;
                }
            }
        }
        const bool in = at >= 0;
        wave_combine_add<4>(in, off, geo, S.d_color + grad_copy(S) + (in ? off : 0));
        wave_combine_add<2>(in, off + 4 + at, offs, S.d_color + grad_copy(S) + (in ? off + 4 + at : 0));
        wave_combine_add<8>(in, off + 4 + ns + 4 * at, cols, S.d_color + grad_copy(S) + (in ? off + 4 + ns + 4 * at : 0));
    }
    float v[4] = {d_color.x, d_color.y, d_color.z, d_color.w};
    wave_combine_add<4>(full >= 0, full, v, S.d_color + grad_copy(S) + (full >= 0 ? full : 0));
}

// d_compute_distance for a whole wave (every lane calls it; lanes without a distance
// adjoint pass active = false): the values of the per-lane version, with the point,
// shape-parameter and transform adjoints of lanes that share a segment, shape or group
// added together before the atomics.  A distance field or a prefiltered image of a few
// shapes sends nearly every sample's adjoint to the same dozen addresses.
DVG_DEV void d_compute_distance_wave(const DevScene &S, bool active, int g, int s, V2 pt, V2 closest,
                                     const PathInfo &info, float d_dist, float *d_translation) {
    const bool act = active && !(dist_sq(pt, closest) < 1e-10f);
    DistAdj a;
    if (act) {
        d_compute_distance_vals(S, g, s, pt, closest, info, d_dist, a);
    } else {
        a.seg = -1;
        a.npar = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            a.pts.use[j] = false;
            a.pts.idx[j] = 0;
            a.pts.d[j] = V2{0, 0};
            a.par[j] = 0.f;
        }
#pragma unroll
        for (int i = 0; i < 9; i++) a.xform[i] = 0.f;
        a.d_pt = V2{0, 0};
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const bool on = act && a.pts.use[j];
        float v[2] = {a.pts.d[j].x, a.pts.d[j].y};
        wave_combine_add<2>(on, a.seg, v, S.d_points + grad_copy(S) + (on ? 2 * a.pts.idx[j] : 0));
    }
    {
        // circle: radius, centre; rect: p_min, p_max -- contiguous at the shape's offset
        const bool on = act && a.npar > 0;
        wave_combine_add<4>(on, s, a.par, S.d_params + grad_copy(S) + (on ? S.param_off[s] : 0), a.npar);
    }
    wave_combine_add<9>(act, g, a.xform, S.d_xform + grad_copy(S) + (act ? 9 * g : 0));
    if (act && d_translation) aadd2(d_translation, -a.d_pt);
}

// composite_adjoint_prefiltered for a whole wave, lanes in lockstep by fragment position
// (as composite_adjoint_wave): paints, stroke widths and distance adjoints are combined
// across lanes.  Every lane must call it; lanes without fragments pass nf = 0.
DVG_DEV V4 composite_adjoint_prefiltered_wave(const DevScene &S, const PFragRec *frags, int nf, V3 final_color,
                                              float final_alpha, V4 d_color, V2 pt, float *d_translation) {
    V3 d_final_color{d_color.x, d_color.y, d_color.z};
    V3 d_curr_color = d_final_color;
    float d_curr_alpha = d_color.w;
    if (nf > 0 && final_alpha > 1e-6f) {
        d_curr_color = vdiv(d_final_color, final_alpha);
        d_curr_alpha -= vsum(d_final_color * final_color) / final_alpha;
    }
    int mx = nf;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, __shfl_xor(mx, o, 64));
    for (int i = mx - 1; i >= 0; i--) {
        const bool on = i < nf;
        PFragRec f{};
        if (on) f = frags[i];
        int g = 0, s = 0, type = -1, off = 0, ns = 0;
        bool paint_on = false, dist_on = false, sw_on = false;
        float d_d = 0.f, d_sw = 0.f;
        V4 dci{0, 0, 0, 0};
        if (on) {
            float d_prev_alpha = d_curr_alpha * (1.f - f.alpha);
            float d_alpha_i = d_curr_alpha * (1.f - f.prev_alpha);
            d_alpha_i += vsum(d_curr_color * (f.color - f.prev_color));
            V3 d_prev_color = d_curr_color * (1 - f.alpha);
            V3 d_color_i = d_curr_color * f.alpha;
            g = f.gid >> 1;
            s = f.shape_id;
            float d = f.distance;
            if (f.gid & 1) {
                type = S.stroke_type[g];
                off = S.stroke_off[g];
                ns = S.stroke_ns[g];
                float sw = S.stroke_width[s];
                float ad = (float)fabs((double)d);
                float apw = ad + sw, amw = ad - sw;
                float w = smoothstep(apw) - smoothstep(amw);
                if (w != 0) {
                    float d_w = w > 0 ? (f.alpha / w) * d_alpha_i : 0.f;
                    d_alpha_i *= w;
                    paint_on = true;
                    dci = V4{d_color_i.x, d_color_i.y, d_color_i.z, d_alpha_i};
                    float d_apw = d_smoothstep(apw, d_w);
                    float d_amw = -d_smoothstep(amw, d_w);
                    d_d = d_apw + d_amw;
                    if (d < 0) d_d = -d_d;
                    d_sw = d_apw - d_amw;
                    dist_on = fabs((double)d_d) > 1e-10f;
                    sw_on = true;
                }
            } else {
                type = S.fill_type[g];
                off = S.fill_off[g];
                ns = S.fill_ns[g];
                float w = smoothstep(d);
                if (w != 0) {
                    float d_w = w > 0 ? (f.alpha / w) * d_alpha_i : 0.f;
                    d_alpha_i *= w;
                    paint_on = true;
                    dci = V4{d_color_i.x, d_color_i.y, d_color_i.z, d_alpha_i};
                    d_d = d_smoothstep(d, d_w);
                    if (d < 0) d_d = -d_d;
                    dist_on = fabs((double)d_d) > 1e-10f && f.within;
                }
            }
            d_curr_color = d_prev_color;
            d_curr_alpha = d_prev_alpha;
        }
        d_sample_paint_wave(S, paint_on, type, off, ns, pt, dci, d_translation);
        d_compute_distance_wave(S, dist_on, g, s, pt, on ? f.closest : pt, f.info, d_d, d_translation);
        {
            float v[1] = {d_sw};
            wave_combine_add<1>(sw_on, s, v, S.d_stroke_width + grad_copy(S) + (sw_on ? s : 0));
        }
    }
    return V4{d_curr_color.x, d_curr_color.y, d_curr_color.z, d_curr_alpha};
}

// composite_adjoint for a whole wave: lanes walk their fragment lists in lockstep by
// position (each lane still goes from its last fragment to its first), so that lanes of
// a tile that see the same paint at the same depth add their constant-paint adjoints
// together before the atomics.  Every lane of the wave must call it; lanes without
// fragments pass nf = 0 and get d_color back.
DVG_DEV V4 composite_adjoint_wave(const DevScene &S, const FragRec *frags, int nf, V3 final_color, float final_alpha,
                                  V4 d_color, V2 pt, float *d_translation) {
    V3 d_final_color{d_color.x, d_color.y, d_color.z};
    V3 d_curr_color = d_final_color;
    float d_curr_alpha = d_color.w;
    if (nf > 0 && final_alpha > 1e-6f) {
        d_curr_color = vdiv(d_final_color, final_alpha);
        d_curr_alpha -= vsum(d_final_color * final_color) / final_alpha;
    }
    int mx = nf;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, __shfl_xor(mx, o, 64));
    for (int i = mx - 1; i >= 0; i--) {
        const bool on = i < nf;
        FragRec f = on ? frags[i] : FragRec{};
        V4 dci{0, 0, 0, 0};
        int g = 0, type = -1, off = 0, ns = 0;
        if (on) {
            g = f.gid >> 1;
            if (f.gid & 1) {
                type = S.stroke_type[g];
                off = S.stroke_off[g];
                ns = S.stroke_ns[g];
            } else {
                type = S.fill_type[g];
                off = S.fill_off[g];
                ns = S.fill_ns[g];
            }
            const V4 c = sample_paint(S, type, off, ns, pt);
            float d_prev_alpha = d_curr_alpha * (1.f - c.w);
            float d_alpha_i = d_curr_alpha * (1.f - f.prev_alpha);
            d_alpha_i += vsum(d_curr_color * (V3{c.x, c.y, c.z} - f.prev_color));
            V3 d_prev_color = d_curr_color * (1 - c.w);
            V3 d_color_i = d_curr_color * c.w;
            dci = V4{d_color_i.x, d_color_i.y, d_color_i.z, d_alpha_i};
            d_curr_color = d_prev_color;
            d_curr_alpha = d_prev_alpha;
        }
        d_sample_paint_wave(S, on, type, off, ns, pt, dci, d_translation);
    }
    return V4{d_curr_color.x, d_curr_color.y, d_curr_color.z, d_curr_alpha};
}

}  // namespace dvg
