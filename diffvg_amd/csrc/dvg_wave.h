// dvg_wave.h -- coverage of a wave's sample points by a list of groups, the work shared out
// over the wave's lanes.
//
// Shading one point per lane, each lane walking the segments that its own point must test,
// keeps a third to a half of the lanes busy: a segment is tested by the lanes whose box test
// it passes, and one lane that needs the double-precision solve holds up 63 (k_edge of the
// 300-path scene: 0.42 of the lanes active, 22,500 vector instructions a wave; 2,048 strokes:
// 0.35, 37,500).  Here the tests are work items in LDS queues that the wave empties 64 at a
// time, so every lane has an item whoever its point belongs to:
//   * per candidate group, 64 segments at a time are tested against the wave's bounding box
//     (one lane per segment); for each that is left, the lanes whose point its box holds push
//     (segment, slot, lane);
//   * screen: one item per lane, the float test (dvg_winding_fast.h) that decides most of them;
//   * exact: what the screen left open, one item per lane: the reference's decision
//     (cubic_winding_libm and cubic_roots_cr, quad_within; cubic_stroke_search, which keeps the
//     reference's operations only where their last bits decide: kQuinticLarge).
// Results come back through LDS: winding sums (added; their order does not matter) and
// stroke hits (or-ed) per lane and slot.  kWaveSlots candidates are in flight at once; then
// their fragments are composited in the list's order.
//
// SIDES = 2 shades the two points of a boundary sample, 1e-4 of the canvas to either side of
// it.  The screen then runs once, at the sample's own position, with every margin widened by
// the distance to the points: what it decides holds at both.  Only the rest (the sample's own
// curve, mostly) is tested at each point.  The group's box tests are taken exactly, per
// point; a segment's box test only decides whether its contribution, which the box makes
// zero or a miss, is looked for, and the exact stage takes it again at its own point.
//
// Scenes that qualify: DevScene::wave_ok.
#pragma once

#include "dvg_memory.h"
#include "dvg_query.h"

namespace dvg {

constexpr int kWaveSlots = 8;   // at most 16 (queue entries, hit masks)
constexpr int kWaveList = 256;  // candidates listed at a time

template <int SIDES>
struct WaveLds {
    float2 pt[SIDES][64];       // canvas points
    int wn[kWaveSlots][64];     // winding sums (side 1 in the upper 16 bits)
    int hit[64];                // stroke hits: bit slot + 16 side
    int q1[128];                // screen queue: segment << 10 | slot << 6 | lane
    float q1x[128], q1y[128];   // and the point in the group's space
    int q2[64 + 64 * SIDES];    // exact queue: segment << 11 | side << 10 | slot << 6 | lane
    int list[kWaveList];        // candidate groups, in increasing order
    int group[kWaveSlots], shape[kWaveSlots];
    float hx[kWaveSlots], hy[kWaveSlots];  // how far the sides lie from the middle, in the group's space
};

// The scene descriptor where it lies in memory (a kernel's arguments, a job table), constant
// while the kernel runs.  get() loads it through scalar loads at the point of the call and no
// earlier: a DevScene is some 60 pointers, and with all of them live across the phases of
// wave_shade the compiler keeps over a thousand scalar registers in vector lanes.  What a
// caller does not use of the copy is not loaded.
struct SceneRef {
    uint64_t at;
    DVG_DEV DevScene get() const {
        uint64_t p = at;
        asm volatile("" : "+s"(p));
        return load_constant<DevScene>(p);
    }
};
// of a kernel whose first argument is the DevScene
DVG_DEV SceneRef scene_argument() { return SceneRef{(uint64_t)__builtin_amdgcn_kernarg_segment_ptr()}; }

// segment_within_lq for paths without the approximate quadratic distance
DVG_DEV bool wave_within_lq(const DevScene &S, int s, int seg, int k, V2 pt, float r) {
    V2 p[4];
    int4 idx;
    seg_load(S, seg, p, idx);
    float r0 = r, r1 = r, r2 = r;
    if (S.has_thick[s]) {
        r0 = S.thickness[idx.x];
        r1 = S.thickness[idx.y];
        if (k == 1) r2 = S.thickness[idx.z];
    }
    if (k == 0) return line_within(p[0], p[1], pt, r0, r1);
    return quad_within(p[0], p[1], p[2], pt, r0, r1, r2);
}

// Orders the wave's LDS accesses (a wave's LDS instructions execute in order; this keeps the
// compiler from moving them).
DVG_DEV void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
DVG_DEV int rank_below(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}
DVG_DEV float lane_value(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
DVG_DEV bool is_affine(const M3 &m) { return m.m[6] == 0.f && m.m[7] == 0.f && m.m[8] == 1.f; }
// xform_pt without its division when the last row is (0, 0, 1): the divisor is then exactly 1
DVG_DEV V2 xform_fast(const M3 &m, bool affine, V2 p) {
    if (!affine) return xform_pt(m, p);
    return V2{m.m[0] * p.x + m.m[1] * p.y + m.m[2], m.m[3] * p.x + m.m[4] * p.y + m.m[5]};
}

// The exact stage: the last `cnt` items of the exact queue, one per lane.
template <int SIDES, bool STROKE>
DVG_DEV void wave_exact(const SceneRef &R, WaveLds<SIDES> &W, int &n2, int cnt) {
    const DevScene S = R.get();
    const int lane = threadIdx.x & 63;
    wave_sync();
    n2 -= cnt;
    if (lane < cnt) {
        const unsigned id = (unsigned)W.q2[n2 + lane];
        const int owner = id & 63, slot = (id >> 6) & 15, side = SIDES == 2 ? (id >> 10) & 1 : 0, seg = id >> 11;
        const int g = W.group[slot], s = W.shape[slot];
        const float2 c = W.pt[side][owner];
        const V2 p = xform_pt(m3_load(S.c2s + 9 * g), V2{c.x, c.y});
        const bool one = S.nsegs[s] == 1;
        const int k = S.seg_kind[seg];
        if constexpr (STROKE) {
            const int bit = 1 << (slot + 16 * side);
            if (!(W.hit[owner] & bit) && (one || in_box(S.seg_box[seg], p, S.seg_maxr[seg]))) {
                const float r = S.stroke_width[s];
                bool hit;
                if (k == 2) {
                    const CubicPoints c = cubic_points_of(S, seg);
                    float r0 = r, r1 = r, r2 = r, r3 = r;
                    if (S.has_thick[s]) {
                        const int4 idx = S.seg_idx[seg];
                        r0 = S.thickness[idx.x];
                        r1 = S.thickness[idx.y];
                        r2 = S.thickness[idx.z];
                        r3 = S.thickness[idx.w];
                    }
                    hit = dist_sq(c.p0, p) < r0 * r0 || dist_sq(c.p3, p) < r3 * r3;
                    if (!hit) hit = cubic_stroke_search(cubic_points_at(S, seg), p, r0, r1, r2, r3);
                } else {
                    hit = wave_within_lq(S, s, seg, k, p, r);
                }
                if (hit) atomicOr(&W.hit[owner], bit);
            }
        } else if (one || ray_box(S.seg_box[seg], p)) {
            int w = 0;
            if (k == 2) {
                if (!wf::cubic_winding_test<true>(cubic_prep_of(S, seg), p.x, p.y, w)) {
                    const CubicPoints c = cubic_points_of(S, seg);
                    w = cubic_winding_solve(c.p0, c.p1, c.p2, c.p3, p);
                }
            } else {
                V2 q[4];
                int4 idx;
                seg_load(S, seg, q, idx);
                w = segment_winding_lq(k, q, p);
            }
            if (w) atomicAdd(&W.wn[slot][owner], side ? w * 65536 : w);
        }
    }
    wave_sync();
}

// The screen: the last `cnt` items of the screen queue, one per lane.
template <int SIDES, bool STROKE>
DVG_DEV void wave_screen(const SceneRef &R, WaveLds<SIDES> &W, int &n1, int &n2, int cnt) {
    const DevScene S = R.get();
    const int lane = threadIdx.x & 63;
    wave_sync();
    n1 -= cnt;
    bool open = false;
    unsigned id = 0;
    if (lane < cnt) {
        id = (unsigned)W.q1[n1 + lane];
        const V2 pt{W.q1x[n1 + lane], W.q1y[n1 + lane]};
        const int owner = id & 63, slot = (id >> 6) & 15, seg = id >> 10;
        const float hx = SIDES == 2 ? W.hx[slot] : 0.f, hy = SIDES == 2 ? W.hy[slot] : 0.f;
        const int k = S.seg_kind[seg];
        if constexpr (STROKE) {
            const int s = W.shape[slot];
            constexpr int both = SIDES == 2 ? 0x10001 : 1;
            if ((W.hit[owner] & (both << slot)) != (both << slot)) {
                const float r = S.stroke_width[s];
                if (k == 2) {
                    const wf::StrokePrep q = stroke_prep_of(S, seg);
                    float r0 = r, r3 = r, rmax = fabsf(r);
                    if (S.has_thick[s]) {
                        const int4 idx = S.seg_idx[seg];
                        r0 = S.thickness[idx.x];
                        r3 = S.thickness[idx.w];
                        rmax = fmaxf(fmaxf(fabsf(r0), fabsf(S.thickness[idx.y])),
                                     fmaxf(fabsf(S.thickness[idx.z]), fabsf(r3)));
                    }
                    bool hit;
                    float reach = 0.f;
                    if constexpr (SIDES == 2) {
                        reach = hx + hy;
                        hit = wf::stroke_ends_within(q, pt.x, pt.y, r0, r3, reach);
                    } else {
                        const V2 p0{q.x[0], q.y[0]}, p3{q.x[8], q.y[8]};
                        hit = dist_sq(p0, pt) < r0 * r0 || dist_sq(p3, pt) < r3 * r3;
                    }
                    if (hit) {
                        atomicOr(&W.hit[owner], both << slot);
                    } else {
                        open = !wf::stroke_farther(q, pt.x, pt.y, rmax + reach);
                    }
                } else if constexpr (SIDES == 1) {
                    if (wave_within_lq(S, s, seg, k, pt, r)) atomicOr(&W.hit[owner], both << slot);
                } else {
                    open = true;
                }
            }
        } else {
            int w = 0;
            if (k == 2) {
                open = !wf::cubic_winding_test<false>(cubic_prep_of(S, seg), pt.x, pt.y, w, hx, hy);
            } else if constexpr (SIDES == 1) {
                V2 p[4];
                int4 idx;
                seg_load(S, seg, p, idx);
                w = segment_winding_lq(k, p, pt);
            } else {
                open = true;
            }
            if (!open && w) atomicAdd(&W.wn[slot][owner], SIDES == 2 ? w * 65537 : w);
        }
    }
    const uint64_t m = __ballot(open);
    if (m) {
        const int at = n2 + rank_below(m), c = __popcll(m);
        const int item = (int)(((id >> 10) << 11) | (id & 1023u));
        if (open) {
            W.q2[at] = item;
            if constexpr (SIDES == 2) W.q2[at + c] = item | 1024;
        }
        n2 += SIDES * c;
    }
}

// The winding sums (or stroke hits) of the path candidates `todo` (a bit per slot) at the
// points whose boxes hold them (`in`, wave_shade): pushes their tests, screening whenever 64
// are waiting, until the queues are empty.
template <int SIDES, bool STROKE>
DVG_DEV void wave_paths(const SceneRef &R, WaveLds<SIDES> &W, unsigned todo, unsigned in, V2 pm, float4 wbox) {
    const int lane = threadIdx.x & 63;
    int n1 = 0, n2 = 0;
    // the block of up to 64 segments being pushed: box (grown by the radius, for strokes) of
    // segment j0 + lane, and which of them are left
    float4 box = make_float4(0.f, 0.f, 0.f, 0.f);
    uint64_t left = 0;
    int slot = 0, j0 = 0, nb = 0, sb = 0;
    float hx = 0.f, hy = 0.f, wx0 = 0.f, wy0 = 0.f, wx1 = 0.f, wy1 = 0.f;
    V2 lm{0, 0};
    bool on = false;
    for (;;) {
        while (n1 < 64) {
            if (!left) {
                const DevScene S = R.get();
                j0 += 64;
                if (j0 >= nb) {
                    if (!todo) break;
                    slot = __ffs(todo) - 1;
                    todo &= todo - 1;
                    const int g = __builtin_amdgcn_readfirstlane(W.group[slot]);
                    const int s = __builtin_amdgcn_readfirstlane(W.shape[slot]);
                    if constexpr (SIDES == 2) {
                        hx = lane_value(W.hx[slot], 0);
                        hy = lane_value(W.hy[slot], 0);
                    }
                    const M3 m = m3_load(S.c2s + 9 * g);
                    const bool affine = is_affine(m);
                    lm = xform_fast(m, affine, pm);
                    on = ((in >> slot) & 0x10001u) != 0;
                    // the wave's box in the group's space, widened for rounding
                    wx0 = wy0 = -__builtin_huge_valf();
                    wx1 = wy1 = __builtin_huge_valf();
                    if (affine) {
                        const float cx = 0.5f * (wbox.x + wbox.z), cy = 0.5f * (wbox.y + wbox.w);
                        const float ex = 0.5f * (wbox.z - wbox.x), ey = 0.5f * (wbox.w - wbox.y);
                        const V2 c = xform_fast(m, true, V2{cx, cy});
                        const float mag = 4e-6f * ((fabsf(m.m[0]) + fabsf(m.m[3])) * (fabsf(cx) + ex) +
                                                   (fabsf(m.m[1]) + fabsf(m.m[4])) * (fabsf(cy) + ey) +
                                                   fabsf(m.m[2]) + fabsf(m.m[5]));
                        const float rx = (fabsf(m.m[0]) * ex + fabsf(m.m[1]) * ey) * 1.00001f + mag + hx;
                        const float ry = (fabsf(m.m[3]) * ex + fabsf(m.m[4]) * ey) * 1.00001f + mag + hy;
                        wx0 = c.x - rx, wx1 = c.x + rx, wy0 = c.y - ry, wy1 = c.y + ry;
                    }
                    nb = S.nsegs[s], sb = S.seg_begin[s], j0 = 0;
                }
                const int j = j0 + lane;
                bool keep = false;
                if (j < nb) {
                    box = S.seg_box[sb + j];
                    if constexpr (STROKE) {
                        const float r = S.seg_maxr[sb + j];
                        box = make_float4(box.x - r, box.y - r, box.z + r, box.w + r);
                        keep = nb == 1 || !(wx1 < box.x || wx0 > box.z || wy1 < box.y || wy0 > box.w);
                    } else {
                        keep = nb == 1 || !(wy1 < box.y || wy0 > box.w || wx0 > box.z);
                    }
                }
                left = __ballot(keep);
                continue;
            }
            const int jj = __ffsll((unsigned long long)left) - 1;
            left &= left - 1;
            bool test = on;
            if (nb != 1) {
                // in_box / ray_box of the reference at every point within hx, hy of lm
                const float x0 = lane_value(box.x, jj), y0 = lane_value(box.y, jj), x1 = lane_value(box.z, jj),
                            y1 = lane_value(box.w, jj);
                if constexpr (STROKE)
                    test = on && lm.x + hx >= x0 && lm.x - hx <= x1 && lm.y + hy >= y0 && lm.y - hy <= y1;
                else
                    test = on && !(lm.y + hy < y0 || lm.y - hy > y1) && !(lm.x - hx > x1);
            }
            const uint64_t t = __ballot(test);
            if (test) {
                const int at = n1 + rank_below(t);
                W.q1[at] = (int)(((unsigned)(sb + j0 + jj) << 10) | (unsigned)(slot << 6) | (unsigned)lane);
                W.q1x[at] = lm.x;
                W.q1y[at] = lm.y;
            }
            n1 += __popcll(t);
        }
        const bool last = n1 < 64;  // nothing left to push
        if (n1) wave_screen<SIDES, STROKE>(R, W, n1, n2, min(n1, 64));
        while (n2 >= 64 || (last && n2)) wave_exact<SIDES, STROKE>(R, W, n2, min(n2, 64));
        if (last) break;
    }
}

// Coverage of the wave's points by the listed candidates, in their order (wave_shade).
template <int SIDES, class Emit>
DVG_DEV void wave_candidates(const SceneRef &R, WaveLds<SIDES> &W, int n, bool valid, V2 pa, V2 pb, V2 pm, float cx,
                             float cy, float4 wbox, const Emit &emit) {
    const int lane = threadIdx.x & 63;
    const float inf = __builtin_huge_valf();
    for (int base = 0; base < n; base += kWaveSlots) {
        const int cnt = min(kWaveSlots, n - base);
        // which points each candidate's boxes hold (bit slot + 16 side), and shapes without
        // segments
        unsigned in_s = 0, in_f = 0, paths_s = 0, paths_f = 0;
        for (int k = 0; k < cnt; k++) {
            const DevScene S = R.get();
            const int g = __builtin_amdgcn_readfirstlane(W.list[base + k]);
            const float4 b = S.g_box[g];
            const float mr = S.g_maxr[g];
            const bool a0 = valid && (S.ng == 1 || in_box(b, pa, mr));
            const bool a1 = SIDES == 2 && valid && (S.ng == 1 || in_box(b, pb, mr));
            if (!__any(a0 || a1)) continue;
            const int s = S.g_ids[S.g_off[g]];
            const M3 m = m3_load(S.c2s + 9 * g);
            const bool affine = is_affine(m);
            const int type = S.shape_type[s];
            const bool path = type == 2;
            const bool st = S.stroke_type[g] >= 0, ft = S.fill_type[g] >= 0;
            const V2 la = xform_fast(m, affine, pa);
            V2 lb = la;
            if constexpr (SIDES == 2) lb = xform_fast(m, affine, pb);
            if (lane == 0) {
                W.group[k] = g;
                W.shape[k] = s;
                if constexpr (SIDES == 2) {
                    // half the distance of the sides in the group's space, with 1% and the
                    // rounding of the transforms on top
                    const float mag = 2e-6f * ((fabsf(m.m[0]) + fabsf(m.m[3])) * S.cw +
                                               (fabsf(m.m[1]) + fabsf(m.m[4])) * S.ch + fabsf(m.m[2]) + fabsf(m.m[5]));
                    W.hx[k] = affine ? fabsf(m.m[0]) * cx + fabsf(m.m[1]) * cy + mag : inf;
                    W.hy[k] = affine ? fabsf(m.m[3]) * cx + fabsf(m.m[4]) * cy + mag : inf;
                }
            }
            if (st) {
                if (path) {
                    in_s |= (a0 ? 1u << k : 0u) | (a1 ? 0x10000u << k : 0u);
                    paths_s |= 1u << k;
                } else {
                    const float r = S.stroke_width[s];
                    const bool h0 = a0 && within_distance_prim(S, s, type, la, r);
                    const bool h1 = a1 && within_distance_prim(S, s, type, lb, r);
                    if (h0 || h1) W.hit[lane] |= (h0 ? 1 << k : 0) | (h1 ? 0x10000 << k : 0);
                    in_s |= (a0 ? 1u << k : 0u) | (a1 ? 0x10000u << k : 0u);
                }
            }
            if (ft) {
                const float4 lbox = S.g_lbox[g];
                const bool f0 = a0 && in_box(lbox, la), f1 = a1 && in_box(lbox, lb);
                in_f |= (f0 ? 1u << k : 0u) | (f1 ? 0x10000u << k : 0u);
                if (path) {
                    if (__any(f0 || f1)) paths_f |= 1u << k;
                } else {
                    const int w0 = f0 ? winding_prim(S, s, type, la) : 0, w1 = f1 ? winding_prim(S, s, type, lb) : 0;
                    W.wn[k][lane] = w0 + (SIDES == 2 ? w1 * 65536 : 0);
                }
            }
        }
        wave_sync();
        if (paths_f) wave_paths<SIDES, false>(R, W, paths_f, in_f, pm, wbox);
        if (paths_s) wave_paths<SIDES, true>(R, W, paths_s, in_s, pm, wbox);
        wave_sync();
        const unsigned hits = (unsigned)W.hit[lane] & in_s;
        W.hit[lane] = 0;
        // a candidate's stroke (even steps), then its fill
        for (int i = 0; i < 2 * cnt; i++) {
            const int k = i >> 1;
            const bool stroke = !(i & 1);
            const unsigned in = (stroke ? hits : in_f) >> k;
            bool a = (in & 1u) != 0, b = (in & 0x10000u) != 0;
            if (!__any(a || b)) continue;
            const DevScene S = R.get();
            const int g = __builtin_amdgcn_readfirstlane(W.group[k]);
            if (!stroke) {
                const int v = W.wn[k][lane];
                W.wn[k][lane] = 0;
                const int w0 = SIDES == 2 ? (int)(short)(v & 0xffff) : v;
                const int w1 = SIDES == 2 ? (v - w0) >> 16 : 0;
                const bool eo = S.even_odd[g] != 0;
                a = a && (eo ? (w0 & 1) != 0 : w0 != 0);
                b = b && (eo ? (w1 & 1) != 0 : w1 != 0);
            }
            if (__any(a || b)) emit(S, g, stroke, a, b);
        }
        wave_sync();
    }
}

// Coverage of the wave's points by the scene's groups, in increasing order: emit(S, g, stroke,
// a, b) for every group and paint that covers some lane's point (stroke before fill of a
// group), a and b whether it covers this lane's first and second point.  Every lane of the
// wave calls it; lanes without a point pass valid = false.  pm: the point the screen uses
// (SIDES = 1: pa itself); cx, cy: bounds on |pa - pm| and |pb - pm| per canvas coordinate.
// Each wave lists its own candidates, the groups whose inflated top-level box meets the box
// of its points, so waves do not wait for each other and a wave of 64 samples tests a
// smaller box than a tile of 256.
template <int SIDES, class Emit>
DVG_DEV void wave_shade(const SceneRef &R, WaveLds<SIDES> &W, bool valid, V2 pa, V2 pb, V2 pm, float cx, float cy,
                        const Emit &emit) {
    const int lane = threadIdx.x & 63;
    W.pt[0][lane] = make_float2(pa.x, pa.y);
    if constexpr (SIDES == 2) W.pt[1][lane] = make_float2(pb.x, pb.y);
    W.hit[lane] = 0;
#pragma unroll
    for (int k = 0; k < kWaveSlots; k++) W.wn[k][lane] = 0;
    const float inf = __builtin_huge_valf();
    float4 wbox = valid ? make_float4(pm.x, pm.y, pm.x, pm.y) : make_float4(inf, inf, -inf, -inf);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        wbox.x = fminf(wbox.x, __shfl_xor(wbox.x, o, 64));
        wbox.y = fminf(wbox.y, __shfl_xor(wbox.y, o, 64));
        wbox.z = fmaxf(wbox.z, __shfl_xor(wbox.z, o, 64));
        wbox.w = fmaxf(wbox.w, __shfl_xor(wbox.w, o, 64));
    }
    int g0 = 0, ng;
    do {
        int n = 0;
        {
            const DevScene S = R.get();
            ng = S.ng;
            for (; g0 < ng && n <= kWaveList - 64; g0 += 64) {
                const int g = g0 + lane;
                bool hit = false;
                if (g < ng) {
                    const float4 b = S.g_box[g];
                    const float r = S.g_maxr[g];
                    // a single group is the root of the top-level BVH and is visited untested
                    hit = ng == 1 || !(b.x - r > wbox.z + cx || b.z + r < wbox.x - cx || b.y - r > wbox.w + cy ||
                                       b.w + r < wbox.y - cy);
                }
                const uint64_t m = __ballot(hit);
                if (hit) W.list[n + rank_below(m)] = g;
                n += __popcll(m);
            }
        }
        wave_sync();
        wave_candidates<SIDES>(R, W, n, valid, pa, pb, pm, cx, cy, wbox, emit);
    } while (g0 < ng);
}

}  // namespace dvg
