// Variable-width stroke (StrokeOptions::variable_line_width) for gfx950.
//
// lyon's second stroker (stroke.rs:653-767, 1380-1512): every endpoint carries a width
// factor (a custom attribute), curves interpolate it, and each edge gets its own side lines
// (tangent to its two end circles), from which every join finds its sides.
//
// The walk is made parallel by what a step really carries over:
//   * which points are kept depends on positions alone (a point too close to the last
//     buffered one is dropped), and the last buffered point is always the newest kept one;
//   * the running length (`advancement`) is a serial f32 sum of the kept edges' lengths;
//   * an edge's side lines depend on its two end points, a join's sides on the side lines
//     of the edges before and after it;
//   * ids are prefix sums of what the joins before emit.
// So a batch runs as a pipeline over all points of all paths:
//   vw_plan_kernel    wave per path: flattened points, windows, sub-paths
//   vw_points_kernel  wave per path: the kept points (position, half width, running length)
//   vw_att_kernel     lane per edge next to an endpoint: its side lines' normals (asin, cos
//                     and sin in f64, gathered so that no lane idles)
//   vw_window_kernel  wave per 63 joins: counts, then (second launch) vertices and triangles
//   vw_tail_kernel    lane per sub-path: its end (caps or the closing joins)
// The rare steps that reach further back are taken out of the common path: a join that
// folds back and is skipped (stroke.rs:1784-1788) is found by the count, settled by
// vw_skip_kernel and its windows counted again; MiterClip joins (a clipped side feeds the
// next join's side line, without bound) and paths not as lyon's builders make them go
// through the serial kernel, one lane per path.
//
// The batched stroke workload with a width factor per point (10,000 paths, 81 M points,
// 164.6 M triangles): 10.5 ms per pass, of which the kept points 2.6 ms, the count 2.3 ms and
// the emission 4.8 ms; one lane per path for the whole walk took 1,059 ms, bound by the
// latency of one lane's chain.  The output cannot be written in less than 0.7 ms.
#include <hip/hip_runtime.h>

#include "lyg_math.h"
#include "lyg_types.h"
#include "stroke_core.h"
#include "stroke_decode.h"
#include "wave.h"

namespace lyg {

namespace vw {

static constexpr uint32_t MAX_CURVE_POINTS = 1u << 22;  // per curve; more: LYG_ERR_NO_SPACE

struct Side {
    vec2 prev, next, single;
    uint32_t prev_v, next_v;
    bool has_single;
};
// EndpointData (stroke.rs:320-352) without the vertex source
struct Pt {
    vec2 pos;
    float hw, adv;
    int join;
    Side sp[2];
    bool fold[2];
    bool flat;
    // VertexSource: endpoint (point index sf) or the point at st on the edge sf -> sto
    uint32_t sf, sto;
    float st;
    bool sedge;
};

__device__ __forceinline__ void pt_init(Pt& e, vec2 pos, float hw, int join, bool flat) {
    const float nan = __builtin_nanf("");
    e.sf = e.sto = 0;
    e.st = 0.0f;
    e.sedge = false;
    e.pos = pos;
    e.hw = hw;
    e.adv = nan;
    e.join = join;
    e.flat = flat;
    for (int k = 0; k < 2; ++k) {
        e.sp[k].prev = e.sp[k].next = mk(nan, nan);
        e.sp[k].single = mk(0.0f, 0.0f);
        e.sp[k].prev_v = e.sp[k].next_v = INVALID_ID;
        e.sp[k].has_single = false;
        e.fold[k] = false;
    }
}

struct Stroker {
    float lw, tol, miter_limit, merge2;
    uint32_t start_cap, end_cap, line_join;
    Sink* s;
    vec2 on_path;  // StrokeVertexData: position_on_path, half_width
    float vhw;
    Pt buf[3];     // PointBuffer (stroke.rs:2371-2457), oldest first: buf[count - 1] is last
    uint32_t count;
    Pt firsts[2];
    uint32_t n_firsts;
    bool may_need_empty_cap;
    float sub_path_start_adv;
    uint32_t status;
    // interpolated attributes (emit pass, when asked for): the current vertex source and
    // the first vertex id not yet given its row
    const float* attrs;
    uint32_t n_attrs;
    float* attr_out;  // row of the path's first vertex
    uint32_t sf, sto, filled;
    float st;
    bool sedge;
};

// StrokeVertex::interpolated_attributes (stroke.rs:2728-2746) for the vertices emitted
// since the last source change, then the new source (where lyon sets vertex.src).
__device__ __forceinline__ void flush_attrs(Stroker& S) {
    if (!S.attr_out) return;
    const Sink& k = *S.s;
    for (uint32_t v = S.filled; v < k.vid; ++v) {
        const uint32_t row = v - k.vid0;
        if (row >= k.vlim) break;
        const float* a = S.attrs + (size_t)S.sf * S.n_attrs;
        const float* b = S.attrs + (size_t)S.sto * S.n_attrs;
        float* o = S.attr_out + (size_t)row * S.n_attrs;
        for (uint32_t q = 0; q < S.n_attrs; ++q)
            o[q] = S.sedge ? a[q] * (1.0f - S.st) + b[q] * S.st : a[q];
    }
    S.filled = k.vid;
}
__device__ __forceinline__ void set_src(Stroker& S, const Pt& p) {
    flush_attrs(S);
    S.sf = p.sf;
    S.sto = p.sto;
    S.st = p.st;
    S.sedge = p.sedge;
}

// Slots are addressed with constant indices only (the step is instantiated per count), so
// the points stay in registers.
template <uint32_t C>
__device__ __forceinline__ void push_n(Stroker& S, const Pt& p) {
    if (C < 3) {
        S.buf[C < 3 ? C : 2] = p;
        S.count = C + 1;
    } else {
        S.buf[0] = S.buf[1];
        S.buf[1] = S.buf[2];
        S.buf[2] = p;
    }
}
__device__ __forceinline__ uint32_t vtx(Stroker& S, vec2 normal) {
    return sink_sv(*S.s, S.on_path, normal, S.vhw);
}

// stroke.rs:1869-1904
__device__ __forceinline__ void edge_tris(Stroker& S, const Pt& p0, const Pt& p1) {
    uint32_t p0n = p0.sp[SN].next_v, p0p = p0.sp[SP].next_v;
    uint32_t p1n = p1.sp[SN].prev_v, p1p = p1.sp[SP].prev_v;
    if (p0.fold[SP]) p0n = p0.sp[SP].prev_v;
    if (p0.fold[SN]) p0p = p0.sp[SN].prev_v;
    if (p1.fold[SP]) p1n = p1.sp[SP].next_v;
    if (p1.fold[SN]) p1p = p1.sp[SN].next_v;
    if (p0n == p1p) return;
    if (p0n != p0p && p0p != p1p) sink_tri(*S.s, p0n, p0p, p1p);
    if (p0n != p1n && p1p != p1n) sink_tri(*S.s, p0n, p1p, p1n);
}

// stroke.rs:1968-2021
__device__ __forceinline__ void round_join(Stroker& S, Pt& j, int side) {
    const float PI = 3.14159265358979323846f;
    vec2 sn = sub(j.sp[side].prev, j.pos), en = sub(j.sp[side].next, j.pos);
    uint32_t sv = j.sp[side].prev_v, ev = j.sp[side].next_v;
    const float sign = side == SN ? 1.0f : -1.0f;
    float a0 = angle_of(sn);
    float diff = angle_to(a0, angle_of(en));
    if (diff * sign < 0.0f) diff = sign * (2.0f * PI - ffabs(diff));
    float a1 = a0 + diff;
    if (side == SN) {
        float ta = a0;
        a0 = a1;
        a1 = ta;
        uint32_t tv = sv;
        sv = ev;
        ev = tv;
    }
    tessellate_arc(a0, a1, sv, ev, arc_subdivisions(diff, j.hw, S.tol), S.on_path, S.vhw, *S.s);
}

// stroke.rs:1907-1965
__device__ __forceinline__ void join_tris(Stroker& S, Pt& j) {
    const bool need0 = !j.sp[SP].has_single && !j.fold[SN];
    const bool need1 = !j.sp[SN].has_single && !j.fold[SP];
    const Side &P = j.sp[SP], &N = j.sp[SN];
    if (!j.fold[SP] && !j.fold[SN]) {
        if (need0 && need1) {
            sink_tri(*S.s, P.prev_v, P.next_v, N.next_v);
            sink_tri(*S.s, P.prev_v, N.next_v, N.prev_v);
        } else if (!need0 && need1) {
            sink_tri(*S.s, N.prev_v, P.prev_v, N.next_v);
        } else if (need0 && !need1) {
            sink_tri(*S.s, N.prev_v, P.prev_v, P.next_v);
        }
    }
    if (j.join == LYG_JOIN_ROUND) {
        if (need0) round_join(S, j, SP);
        if (need1) round_join(S, j, SN);
    }
}

// stroke.rs:2024-2055
__device__ __forceinline__ void base_vertices(Stroker& S, Pt& j, int side) {
    Side& sp = j.sp[side];
    if (sp.has_single) {
        uint32_t id = vtx(S, divs(sub(sp.single, j.pos), j.hw));
        sp.prev_v = sp.next_v = id;
    } else {
        uint32_t a = vtx(S, divs(sub(sp.prev, j.pos), j.hw));
        uint32_t b = vtx(S, divs(sub(sp.next, j.pos), j.hw));
        sp.prev_v = a;
        sp.next_v = b;
    }
}

// stroke.rs:1743-1806; true: the join folds back and is skipped
__device__ __forceinline__ bool flattened_step(Stroker& S, Pt& prev, Pt& j, Pt& next) {
    vec2 pe = sub(j.pos, prev.pos);
    float pl = vlen(pe);
    vec2 pt = divs(pe, pl);
    vec2 ne = sub(next.pos, j.pos);
    float nl = vlen(ne);
    vec2 nt = divs(ne, nl);
    vec2 n = compute_normal(pt, nt);
    if (j.adv != j.adv) j.adv = prev.adv + pl;
    if (next.adv != next.adv) next.adv = j.adv + nl;
    vec2 p0 = add(j.pos, mul(n, S.vhw));
    vec2 p1 = sub(j.pos, mul(n, S.vhw));
    j.sp[SP].prev = j.sp[SP].next = j.sp[SP].single = p0;
    j.sp[SP].has_single = true;
    j.sp[SN].prev = j.sp[SN].next = j.sp[SN].single = p1;
    j.sp[SN].has_single = true;
    vec2 v0 = sub(p0, prev.sp[SP].next), v1 = sub(p1, prev.sp[SN].next);
    if (dot(pe, v0) < 0.0f && dot(pe, v1) < 0.0f) return true;
    uint32_t a = vtx(S, n);
    uint32_t b = vtx(S, neg(n));
    j.sp[SP].prev_v = j.sp[SP].next_v = a;
    j.sp[SN].prev_v = j.sp[SN].next_v = b;
    return false;
}

// stroke.rs:1809-1866: side lines of the edge p0 -> p1, tangent to both end circles
__device__ __forceinline__ void attachments(Pt& p0, Pt& p1) {
    const float PI = 3.14159265358979323846f;
    vec2 e = sub(p1.pos, p0.pos);
    float d = vlen(e);
    float ea = angle_of(e);
    float va = (float)asin((double)((p1.hw - p0.hw) / d));
    if (va != va) va = 0.0f;
    for (int side = 0; side < 2; ++side) {
        float nl = side == SN ? -1.0f : 1.0f;
        float na = ea + nl * (PI * 0.5f + va);
        vec2 n = mk(t_cos(na), t_sin(na));
        p0.sp[side].next = add(p0.pos, mul(n, p0.hw));
        p1.sp[side].prev = add(p1.pos, mul(n, p1.hw));
    }
    if (p1.adv != p1.adv) p1.adv = p0.adv + d;
}

// stroke.rs:2060-2128
__device__ __forceinline__ void join_side(const Pt& prev, Pt& j, const Pt& next, float ml,
                                          int side) {
    const float sign = side == SN ? -1.0f : 1.0f;
    vec2 v0 = normalize(sub(j.sp[side].prev, prev.sp[side].next));
    vec2 v1 = normalize(sub(next.sp[side].prev, j.sp[side].next));
    bool inward = cross(v0, v1) * sign > 0.0f;
    bool forward = dot(v0, v1) > 0.0f;
    vec2 n = mul(compute_normal(v0, v1), sign);
    vec2 pv0 = normalize(sub(j.pos, prev.pos));
    vec2 pv1 = normalize(sub(next.pos, j.pos));
    bool same_side = dot(add(v0, v1), add(pv0, pv1)) >= 0.0f;
    if (inward && !forward && same_side) {
        vec2 en = mul(n, j.hw);
        float pl = j.adv - prev.adv;
        float nl = next.adv - j.adv;
        float dn = dot(en, v1) - nl;
        float dp = dot(en, neg(v0)) - pl;
        if (ffmin(dn, dp) > 0.0f || sqlen(n) < 1e-5f) j.fold[side] = true;
    }
    bool concave = inward && same_side && !j.fold[side];
    bool miter = j.join == LYG_JOIN_MITER || j.join == LYG_JOIN_MITER_CLIP;
    if (concave || (miter && !(sqlen(n) > ml * ml * 4.0f))) {
        j.sp[side].has_single = true;
        j.sp[side].single = add(j.pos, mul(n, j.hw));
    } else if (j.join == LYG_JOIN_MITER_CLIP) {
        vec2 n0 = sub(j.sp[side].prev, j.pos), n1 = sub(j.sp[side].next, j.pos);
        vec2 i0, i1;
        clip_intersections(n0, n1, n, ml * j.hw, &i0, &i1);
        j.sp[side].prev = add(j.pos, i0);
        j.sp[side].next = add(j.pos, i1);
    }
}

// step_impl (stroke.rs:1380-1512) with C points buffered; returns whether the point was
// added
template <uint32_t C>
__device__ __forceinline__ bool step_n(Stroker& S, Pt next) {
    if (C > 0) {
        Pt& lp = S.buf[C > 0 ? C - 1 : 0];
        vec2 d = sub(lp.pos, next.pos);
        if (sqlen(d) < S.merge2) {
            if (C == 1) S.may_need_empty_cap = true;
            return false;
        }
        if (!lp.flat || !next.flat) attachments(lp, next);
    }
    bool skip = false;
    if (C > 1) {
        Pt& prev = S.buf[C > 1 ? C - 2 : 0];
        Pt& j = S.buf[C > 1 ? C - 1 : 0];
        set_src(S, j);
        S.on_path = j.pos;
        S.vhw = j.hw;
        bool fast = false;
        if (j.flat) fast = dot(sub(j.pos, prev.pos), sub(next.pos, j.pos)) > 0.0f;
        if (fast) {
            j.join = LYG_JOIN_MITER;
            skip = flattened_step(S, prev, j, next);
        } else {
            join_side(prev, j, next, S.miter_limit, SP);
            join_side(prev, j, next, S.miter_limit, SN);
            if (j.sp[SP].has_single) j.fold[SN] = false;
            if (j.sp[SN].has_single) j.fold[SP] = false;
            base_vertices(S, j, SN);
            base_vertices(S, j, SP);
        }
        if (!skip) {
            if (C > 2) edge_tris(S, prev, j);
            join_tris(S, j);
            if (C == 2) {
                S.firsts[0] = prev;
                S.firsts[1] = j;
                S.n_firsts = 2;
            }
        }
    }
    if (skip) S.buf[C > 0 ? C - 1 : 0] = next;  // replace_last
    else push_n<C>(S, next);
    return true;
}
__device__ __forceinline__ bool step(Stroker& S, const Pt& next) {
    switch (S.count) {
        case 0: return step_n<0>(S, next);
        case 1: return step_n<1>(S, next);
        case 2: return step_n<2>(S, next);
        default: return step_n<3>(S, next);
    }
}

// stroke.rs:2459-2524
__device__ __forceinline__ void round_cap(Stroker& S, vec2 center, float radius, vec2 sn,
                                       uint32_t sv, uint32_t ev, vec2 edge_n, bool is_start) {
    if (radius < S.tol) return;
    float a0 = angle_of(sn);
    float diff = angle_to(a0, angle_of(edge_n));
    float mid = a0 + diff;
    float a1 = mid + diff;
    uint32_t nsub = arc_subdivisions(diff, radius, S.tol);
    S.on_path = center;
    S.vhw = radius;
    uint32_t mv = vtx(S, normalize(edge_n));
    sink_tri(*S.s, sv, mv, ev);
    tessellate_arc(a0, mid, sv, mv, nsub, center, radius, *S.s);
    tessellate_arc(mid, a1, mv, ev, nsub, center, radius, *S.s);
}

// stroke.rs:1282-1316, 2526-2609
__device__ __forceinline__ void empty_cap(Stroker& S) {
    Pt& p = S.buf[0];
    set_src(S, p);
    S.vhw = p.hw;
    S.on_path = p.pos;
    if (S.start_cap == LYG_CAP_SQUARE) {
        uint32_t a = vtx(S, mk(1.0f, 1.0f));
        uint32_t b = vtx(S, mk(1.0f, -1.0f));
        uint32_t c = vtx(S, mk(-1.0f, -1.0f));
        uint32_t d = vtx(S, mk(-1.0f, 1.0f));
        sink_tri(*S.s, a, b, c);
        sink_tri(*S.s, a, c, d);
    } else if (S.start_cap == LYG_CAP_ROUND) {
        const vec2 center = p.pos;
        const float r = S.vhw;
        uint32_t l = vtx(S, mk(-1.0f, 0.0f));
        uint32_t rr = vtx(S, mk(1.0f, 0.0f));
        round_cap(S, center, r, mk(-1.0f, 0.0f), l, rr, mk(0.0f, 1.0f), true);
        round_cap(S, center, r, mk(1.0f, 0.0f), rr, l, mk(0.0f, -1.0f), false);
    }
}

// stroke.rs:2130-2206
__device__ __forceinline__ void last_edge(Stroker& S, const Pt& p0, Pt& p1, bool is_first) {
    vec2 v = sub(p1.pos, p0.pos);
    p1.adv = p0.adv + vlen(v);
    set_src(S, p1);
    S.on_path = p1.pos;
    S.vhw = p1.hw;
    for (int side = 0; side < 2; ++side) {
        vec2 sp = p1.sp[side].prev;
        if (S.end_cap != LYG_CAP_ROUND) {
            float clip = S.end_cap == LYG_CAP_SQUARE ? p1.hw : 0.0f;
            vec2 n = normalize(sub(p1.pos, p0.pos));
            vec2 inter;
            if (!line_isect(add(p1.pos, mul(n, clip)), perp(n), sp, sub(sp, p0.sp[side].next),
                            &inter))
                inter = p1.sp[side].prev;
            p1.sp[side].prev = inter;
        }
        p1.sp[side].prev_v = vtx(S, divs(sub(p1.sp[side].prev, p1.pos), p1.hw));
    }
    if (!is_first) edge_tris(S, p0, p1);
    if (S.end_cap == LYG_CAP_ROUND)
        round_cap(S, p1.pos, p1.hw, sub(p1.sp[SP].prev, p1.pos), p1.sp[SP].prev_v,
                  p1.sp[SN].prev_v, v, false);
}

// stroke.rs:2208-2276
__device__ __forceinline__ void first_edge(Stroker& S, Pt& f, const Pt& second) {
    set_src(S, f);
    S.on_path = f.pos;
    S.vhw = f.hw;
    for (int side = 0; side < 2; ++side) {
        vec2 sp = f.sp[side].next;
        if (S.start_cap != LYG_CAP_ROUND) {
            float clip = S.start_cap == LYG_CAP_SQUARE ? f.hw : 0.0f;
            vec2 n = normalize(sub(f.pos, second.pos));
            vec2 inter;
            if (!line_isect(add(f.pos, mul(n, clip)), perp(n), sp,
                            sub(sp, second.sp[side].prev), &inter))
                inter = f.sp[side].next;
            sp = inter;
        }
        f.sp[side].next_v = vtx(S, divs(sub(sp, f.pos), f.hw));
    }
    edge_tris(S, f, second);
    if (S.start_cap == LYG_CAP_ROUND)
        round_cap(S, f.pos, f.hw, sub(f.sp[SN].next, f.pos), f.sp[SN].next_v, f.sp[SP].next_v,
                  sub(f.pos, second.pos), true);
}

// stroke.rs:1322-1378
__device__ __forceinline__ void end_with_caps(Stroker& S) {
    if (S.may_need_empty_cap && S.count == 1) {
        empty_cap(S);
        return;
    }
    if (S.count >= 2) {
        Pt p0 = S.count == 2 ? S.buf[0] : S.buf[1];
        Pt p1 = S.count == 2 ? S.buf[1] : S.buf[2];
        last_edge(S, p0, p1, S.count == 2);
        S.sub_path_start_adv = p1.adv;
        if (S.count > 2) {
            p0 = S.firsts[0];
            p1 = S.firsts[1];
        }
        first_edge(S, p0, p1);
    }
}

// stroke.rs:1206-1279
__device__ __forceinline__ void close_sub(Stroker& S) {
    if (S.count == 1) empty_cap(S);
    if (S.count <= 2) return;
    Pt p = S.firsts[0];
    p.adv = __builtin_nanf("");
    if (!step(S, p)) S.buf[2].pos = p.pos;
    if (S.n_firsts >= 2) {
        step(S, S.firsts[1]);
        // here count is 3: both steps kept or replaced a point after the two firsts
        Pt& p0 = S.buf[1];
        Pt& p1 = S.buf[2];
        set_src(S, p0);
        S.on_path = p0.pos;
        S.vhw = p0.hw;
        for (int side = 0; side < 2; ++side) {
            vec2 sp = p0.sp[side].has_single ? p0.sp[side].single : p0.sp[side].next;
            p0.sp[side].next_v = vtx(S, divs(sub(sp, p0.pos), p0.hw));
        }
        edge_tris(S, p0, p1);
    }
}

// stroke.rs:1179-1193
__device__ __forceinline__ void end_sub(Stroker& S, bool close) {
    S.may_need_empty_cap = S.may_need_empty_cap || (close && S.count == 1);
    if (close && S.count > 2) close_sub(S);
    else end_with_caps(S);
    S.count = 0;
    S.n_firsts = 0;
}

// One flattened curve piece (half `b` of a split quadratic, or the whole curve): its
// points with the half width interpolated at their t on the whole curve
// (t_whole = t0 + t * t_scale), as quadratic_bezier_to / cubic_bezier_to do.
__device__ __forceinline__ void curve_piece(Stroker& S, const VRec& r, bool b, bool cubic,
                                            float t0, float t_scale, float w0, float w1,
                                            uint32_t id0, uint32_t id1) {
    const uint32_t n = b ? r.nB : r.nA;
    const float stp = b ? r.sB : r.sA;
    if (n > MAX_CURVE_POINTS) {
        S.status = LYG_ERR_NO_SPACE;
        return;
    }
    float t = 0.0f;
    for (uint32_t k = 0; k < n; ++k) {
        vec2 pos;
        float t1;
        if (k + 1 == n) {
            pos = b ? r.toB : r.toA;
            t1 = 1.0f;
        } else {
            t = t + stp;
            t1 = t;
            pos = horner(r, b, cubic && !b, t);
        }
        const float tw = t_scale == 1.0f && t0 == 0.0f ? t1 : t0 + t1 * t_scale;
        Pt e;
        pt_init(e, pos, (w0 * (1.0f - tw) + w1 * tw) * 0.5f, (int)S.line_join, t1 != 1.0f);
        // the endpoint at t == 1, else the edge (stroke.rs:1005-1013, 1041-1050)
        e.sedge = tw != 1.0f;
        e.sf = e.sedge ? id0 : id1;
        e.sto = id1;
        e.st = tw;
        step(S, e);
    }
}

}  // namespace vw


// One lane per path, the first L.paths_per_wave lanes (of a list: as many as the grid needs) of
// each one-wave block taking paths (grid-stride): few paths per wave spread the serial walks over every SIMD and keep the
// lanes of a wave from waiting on each other's branches.  Counting (EMIT false) or writing
// at the scanned offsets.
template <bool EMIT>
__global__ void __launch_bounds__(64) stroke_vw_kernel(StrokeVWLaunch L) {
    using namespace vw;
    const uint32_t n_walk = L.list ? *L.n_list : L.in.n_paths;
    uint32_t ppw = L.paths_per_wave;
    if (L.list) ppw = min((uint32_t)WAVE, max(1u, (n_walk + gridDim.x - 1u) / gridDim.x));
    if (threadIdx.x >= ppw) return;
    for (uint32_t k = blockIdx.x * ppw + threadIdx.x; k < n_walk; k += gridDim.x * ppw) {
        const uint32_t path = L.list ? L.list[k] : k;
        const lyg_stroke_options o = L.opts[L.opts_stride ? path : 0];
        const uint32_t vb = L.in.verb_off[path], ve = L.in.verb_off[path + 1];
        const uint32_t pb = L.in.point_off[path], pe = L.in.point_off[path + 1];
        const float* pts = L.in.points + 2ull * pb;
        const uint32_t npts = pe - pb;
        Sink sk;
        sk.nv = sk.ni = 0;
        sk.emit = EMIT;
        sk.err = L.err;
        if (EMIT) {
            sk.vid = sk.vid0 = L.vertex_offset + L.vtx_off[path];
            sk.vout = L.out_vertices + 2ull * L.vtx_off[path];
            sk.iout = L.out_indices + L.idx_off[path];
            sk.vlim = L.vtx_off[path + 1] - L.vtx_off[path];
            sk.ileft = L.idx_off[path + 1] - L.idx_off[path];
            if (L.path_status[path] != 0) continue;  // the count pass failed it: no output
        } else {
            sk.vid = sk.vid0 = 0;
            sk.vout = nullptr;
            sk.iout = nullptr;
            sk.vlim = sk.ileft = 0;
        }
        Stroker S;
        S.lw = o.line_width;
        S.tol = o.tolerance;
        S.miter_limit = o.miter_limit;
        S.merge2 = ffmax(ffmin(o.tolerance * o.tolerance * 0.5f,
                               o.line_width * o.line_width * 0.05f),
                         1e-8f);  // StrokeBuilderImpl::new (stroke.rs:591-631)
        S.start_cap = o.start_cap;
        S.end_cap = o.end_cap;
        S.line_join = o.line_join;
        S.s = &sk;
        S.on_path = mk(0.0f, 0.0f);
        S.vhw = o.line_width * 0.5f;
        S.count = 0;
        S.n_firsts = 0;
        S.may_need_empty_cap = false;
        S.sub_path_start_adv = 0.0f;
        S.status = 0;
        S.attrs = L.attrs;
        S.n_attrs = L.n_attrs;
        S.attr_out = EMIT && L.out_attrs ? L.out_attrs + (size_t)L.vtx_off[path] * L.n_attrs
                                         : nullptr;
        S.sf = S.sto = 0;
        S.st = 0.0f;
        S.sedge = false;
        S.filled = sk.vid;
        uint32_t cur_id = 0;  // point index (in the batch) of the current endpoint
        auto width = [&](uint32_t i) {
            return i < npts ? L.widths[(size_t)(pb + i) * L.widths_stride]
                            : __builtin_nanf("");
        };
        float cur_w = __builtin_nanf("");
        uint32_t p = 0;
        for (uint32_t v = vb; v < ve && S.status == 0; ++v) {
            const uint8_t verb = L.in.verbs[v];
            VRec r;
            decode_verb(verb, pts, npts, p, o.tolerance, r);
            if (verb == LYG_VERB_BEGIN) {
                cur_w = width(p);
                S.may_need_empty_cap = false;
                Pt e;
                pt_init(e, r.toA, o.line_width * cur_w * 0.5f, (int)o.line_join, false);
                e.adv = S.sub_path_start_adv;
                cur_id = pb + p;
                e.sf = e.sto = cur_id;
                step(S, e);
                p += 1;
            } else if (verb == LYG_VERB_LINE) {
                cur_w = width(p);
                Pt e;
                pt_init(e, r.toA, o.line_width * cur_w * 0.5f, (int)o.line_join, false);
                cur_id = pb + p;
                e.sf = e.sto = cur_id;
                step(S, e);
                p += 1;
            } else if (verb == LYG_VERB_QUADRATIC) {
                const float w0 = o.line_width * cur_w;
                cur_w = width(p + 1);
                const float w1 = o.line_width * cur_w;
                vec2 from = p > 0 ? ldp(pts, npts, p - 1) : mk(__builtin_nanf(""), __builtin_nanf(""));
                const float ts = find_sharp_turn(from, ldp(pts, npts, p), ldp(pts, npts, p + 1));
                const uint32_t id0 = cur_id;
                cur_id = pb + p + 1;
                if (ts > 0.0f) {  // flatten_quad's two halves (stroke.rs:2755-2779)
                    curve_piece(S, r, false, false, 0.0f, ts, w0, w1, id0, cur_id);
                    if (S.status == 0)
                        curve_piece(S, r, true, false, ts, 1.0f - ts, w0, w1, id0, cur_id);
                } else {
                    curve_piece(S, r, false, false, 0.0f, 1.0f, w0, w1, id0, cur_id);
                }
                p += 2;
            } else if (verb == LYG_VERB_CUBIC) {
                const float w0 = o.line_width * cur_w;
                cur_w = width(p + 2);
                const uint32_t id0 = cur_id;
                cur_id = pb + p + 2;
                curve_piece(S, r, false, true, 0.0f, 1.0f, w0, o.line_width * cur_w, id0,
                            cur_id);
                p += 3;
            } else {
                const bool close = verb == LYG_VERB_CLOSE;
                end_sub(S, close);
                if (close) p += 1;
            }
        }
        flush_attrs(S);
        if (!EMIT) {
            const bool ok = S.status == 0;
            L.path_status[path] = S.status;
            L.path_nv[path] = ok ? sk.nv : 0u;
            L.path_ni[path] = ok ? 3u * sk.ni : 0u;
        }
    }
}

// ---- the parallel form -------------------------------------------------------------------
namespace vw {

enum : uint32_t {
    PF_FLAT = 1u,   // inside a curve (is_flattening_step)
    PF_FIRST = 2u,  // first point of its sub-path
    PF_ATT = 4u,    // the edge to this point has side lines (an end of it is an endpoint)
    PF_SKIP = 8u,   // its join folds back and is skipped
    PF_CAND = 16u,  // the count pass found that it might
};
// Joins per window: lane 0 repeats the join before the window (its ids and folds).
static constexpr uint32_t WIN = VW_WINDOW;
static_assert(WIN == WAVE - 1, "lane 0 is the halo");

struct VX {  // per verb of a chunk: line_width * width factor at both ends, split, endpoints
    float w0, w1, ts;
    uint32_t id0, id1;
};

__device__ __forceinline__ void mark_slow(const VWPar& P, uint32_t path) {
    P.path_mode[path] = 1u;
}

// One path's kept points.
struct PC {
    const float4* rec;  // position, half width, running length
    const uint8_t* fl;
    const float4* att;       // side line normals by ordinal
    const uint32_t* win_att; // ordinal of the first edge of every window of the path
    uint32_t kn;
    float tol, ml;
    int join;
};
__device__ __forceinline__ PC path_ctx(const VWPar& P, uint32_t path) {
    const lyg_stroke_options o = P.opts[P.opts_stride ? path : 0];
    PC c;
    c.rec = reinterpret_cast<const float4*>(P.rec) + P.raw_off[path];
    c.fl = P.pflags + P.raw_off[path];
    c.att = reinterpret_cast<const float4*>(P.att_n) + P.att_off[path];
    c.win_att = P.win_att + P.win_off[path];
    c.kn = P.kept_n[path];
    c.tol = o.tolerance;
    c.ml = o.miter_limit;
    c.join = (int)o.line_join;
    return c;
}
__device__ __forceinline__ vec2 pos_of(const float4& r) { return mk(r.x, r.y); }
// The point before point i in the buffer when its own join is processed (i is not FIRST).
__device__ __forceinline__ uint32_t eff_prev(const PC& c, uint32_t i) {
    uint32_t q = i - 1;
    while (c.fl[q] & PF_SKIP) --q;
    return q;
}
// Whether the join at the flat point i takes the fast path (stroke.rs:1427-1432).
__device__ __forceinline__ bool fast_at(const PC& c, uint32_t i) {
    const vec2 p = pos_of(c.rec[eff_prev(c, i)]), j = pos_of(c.rec[i]), n = pos_of(c.rec[i + 1]);
    return dot(sub(j, p), sub(n, j)) > 0.0f;
}
// Ordinal of the first edge with side lines at or after the edge to point i.
__device__ __forceinline__ uint32_t att_ord(const PC& c, uint32_t i) {
    const uint32_t w = i / WIN;
    uint32_t ord = c.win_att[w];
    for (uint32_t k = w * WIN; k < i; ++k) ord += (c.fl[k] & PF_ATT) ? 1u : 0u;
    return ord;
}

// join_side (above) on a join's EPD: the same arithmetic on values.
template <int side>
__device__ __forceinline__ void epd_join_side(EPD& j, vec2 p, vec2 n, vec2 pnext, vec2 nprev,
                                              float hw, float advp, float advj, float advn,
                                              float ml) {
    const float sign = side == SN ? -1.0f : 1.0f;
    const vec2 v0 = normalize(sub(j.prev[side], pnext));
    const vec2 v1 = normalize(sub(nprev, j.next[side]));
    const bool inward = cross(v0, v1) * sign > 0.0f;
    const bool forward = dot(v0, v1) > 0.0f;
    const vec2 nn = mul(compute_normal(v0, v1), sign);
    const vec2 pv0 = normalize(sub(j.pos, p));
    const vec2 pv1 = normalize(sub(n, j.pos));
    const bool same_side = dot(add(v0, v1), add(pv0, pv1)) >= 0.0f;
    if (inward && !forward && same_side) {
        const vec2 en = mul(nn, hw);
        const float pl = advj - advp;
        const float nl = advn - advj;
        const float dn = dot(en, v1) - nl;
        const float dp = dot(en, neg(v0)) - pl;
        if (ffmin(dn, dp) > 0.0f || sqlen(nn) < 1e-5f) j.fold[side] = 1;
    }
    const bool concave = inward && same_side && !j.fold[side];
    // MiterClip paths take the serial kernel
    if (concave || (j.line_join == LYG_JOIN_MITER && !(sqlen(nn) > ml * ml * 4.0f))) {
        j.has_single[side] = 1;
        j.single[side] = add(j.pos, mul(nn, hw));
    }
}

// The join at point i (neither the first nor the last of its sub-path, not skipped), as
// step_n<2 or 3> finds it: J and the buffered point q before it.  `ord` = att_ord(i).
__device__ __forceinline__ void join_at(const PC& c, uint32_t i, uint32_t ord, JInfo& J,
                                        uint32_t& q, bool& pfirst) {
    const float nan = __builtin_nanf("");
    const float4 rj = c.rec[i], rn = c.rec[i + 1];
    const uint32_t fj = c.fl[i], fn = c.fl[i + 1];
    uint32_t before = 0;  // edges with side lines to the skipped points q + 1 .. i - 1
    q = i - 1;
    uint32_t fq = c.fl[q], fq1 = fj;
    while (fq & PF_SKIP) {
        before += (fq & PF_ATT) ? 1u : 0u;
        fq1 = fq;
        --q;
        fq = c.fl[q];
    }
    const float4 rq = c.rec[q];
    pfirst = (fq & PF_FIRST) != 0;
    const vec2 p = pos_of(rq), j = pos_of(rj), n = pos_of(rn);
    const float hw = rj.z;
    const bool flat = (fj & PF_FLAT) != 0;
    J.fast = flat && dot(sub(j, p), sub(n, j)) > 0.0f;
    J.weird = false;
    // the side points q has towards the next point, after its own join
    vec2 pn0 = mk(nan, nan), pn1 = pn0;
    bool fastq = false;
    if (fq & PF_FLAT) {
        const vec2 r = pos_of(c.rec[eff_prev(c, q)]);
        const vec2 nx = q + 1 == i ? j : pos_of(c.rec[q + 1]);
        const vec2 pe = sub(p, r), ne = sub(nx, p);
        fastq = dot(pe, ne) > 0.0f;
        if (fastq) {
            const vec2 nm = compute_normal(divs(pe, vlen(pe)), divs(ne, vlen(ne)));
            pn0 = add(p, mul(nm, rq.z));
            pn1 = sub(p, mul(nm, rq.z));
        }
    }
    if (!fastq && (fq1 & PF_ATT)) {
        const float4 a = c.att[ord - before];
        pn0 = add(p, mul(mk(a.x, a.y), rq.z));
        pn1 = add(p, mul(mk(a.z, a.w), rq.z));
    }
    EPD& x = J.x;
    epd_init(x, j, flat, c.join);
    if (J.fast) {  // flattened_step
        x.line_join = LYG_JOIN_MITER;
        const vec2 pe = sub(j, p), ne = sub(n, j);
        const vec2 nm = compute_normal(divs(pe, vlen(pe)), divs(ne, vlen(ne)));
        J.normal = nm;
        const vec2 p0 = add(j, mul(nm, hw)), p1 = sub(j, mul(nm, hw));
        x.prev[SP] = x.next[SP] = x.single[SP] = p0;
        x.prev[SN] = x.next[SN] = x.single[SN] = p1;
        x.has_single[SP] = x.has_single[SN] = 1;
        J.weird = dot(pe, sub(p0, pn0)) < 0.0f && dot(pe, sub(p1, pn1)) < 0.0f;
    } else {
        vec2 np0 = mk(nan, nan), np1 = np0;
        if (fj & PF_ATT) {
            const float4 a = c.att[ord];
            x.prev[SP] = add(j, mul(mk(a.x, a.y), hw));
            x.prev[SN] = add(j, mul(mk(a.z, a.w), hw));
        }
        if (fn & PF_ATT) {
            const float4 a = c.att[ord + ((fj & PF_ATT) ? 1u : 0u)];
            x.next[SP] = add(j, mul(mk(a.x, a.y), hw));
            x.next[SN] = add(j, mul(mk(a.z, a.w), hw));
            np0 = add(n, mul(mk(a.x, a.y), rn.z));
            np1 = add(n, mul(mk(a.z, a.w), rn.z));
        }
        // Running lengths as they stand when this join is processed.  A flat point after a
        // flat point whose join was not fast has none yet (NaN: no side lines between two
        // flattening steps, no fast path); a fast join fills its own in.
        float advp = rq.w, advj = rj.w;
        if ((fq & PF_FLAT) && !fastq && (c.fl[q - 1] & PF_FLAT) && !fast_at(c, q - 1)) advp = nan;
        if (flat && (c.fl[i - 1] & PF_FLAT) && q + 1 == i && !fastq) advj = nan;
        const float advn = (fn & PF_ATT) ? advj + vlen(sub(n, j)) : nan;
        epd_join_side<SP>(x, p, n, pn0, np0, hw, advp, advj, advn, c.ml);
        epd_join_side<SN>(x, p, n, pn1, np1, hw, advp, advj, advn, c.ml);
        if (x.has_single[SP]) x.fold[SN] = 0;
        if (x.has_single[SN]) x.fold[SP] = 0;
    }
    J.needs[SP] = !x.has_single[SP] && !x.fold[SN];
    J.needs[SN] = !x.has_single[SN] && !x.fold[SP];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        J.arc[side].nsub = 0;
        J.arc[side].a0 = J.arc[side].a1 = 0.0f;
        J.arc[side].swap = side == SN;
        if (x.line_join != LYG_JOIN_ROUND || !J.needs[side]) continue;
        // round_join (above) up to the arc
        const float PI = 3.14159265358979323846f;
        const float sign = side == SN ? 1.0f : -1.0f;
        const float a0 = angle_of(sub(x.prev[side], j));
        float diff = angle_to(a0, angle_of(sub(x.next[side], j)));
        if (diff * sign < 0.0f) diff = sign * (2.0f * PI - ffabs(diff));
        const float a1 = a0 + diff;
        J.arc[side].a0 = side == SN ? a1 : a0;
        J.arc[side].a1 = side == SN ? a0 : a1;
        J.arc[side].nsub = arc_subdivisions(diff, hw, c.tol);
    }
}

// The path's sub-path that point i belongs to (sub-paths in order of their first points).
__device__ __forceinline__ VWTail* tail_of(const VWPar& P, uint32_t path, uint32_t i) {
    uint32_t lo = P.tail_off[path], hi = P.tail_off[path + 1] - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (P.tails[mid].first <= i) lo = mid;
        else hi = mid - 1;
    }
    return P.tails + lo;
}

}  // namespace vw

// Wave per path: flattened points, sub-paths and the edges that may need side lines.  A path
// whose verbs are not Begin (Line | Quadratic | Cubic)* (End | Close) sub-paths, or with
// MiterClip joins, is left to the serial kernel; one with a curve beyond MAX_CURVE_POINTS
// gets its status here.
__global__ void __launch_bounds__(64) vw_plan_kernel(VWPar P) {
    using namespace vw;
    const int l = lane_id();
    for (uint32_t path = blockIdx.x; path < P.in.n_paths; path += gridDim.x) {
        const lyg_stroke_options o = P.opts[P.opts_stride ? path : 0];
        const uint32_t vb = P.in.verb_off[path], nverbs = P.in.verb_off[path + 1] - vb;
        const uint32_t pb = P.in.point_off[path], npts = P.in.point_off[path + 1] - pb;
        const float* pts = P.in.points + 2ull * pb;
        bool bad = o.line_join == LYG_JOIN_MITER_CLIP, space = false, open = false;
        uint64_t raw = 0;
        uint32_t ends = 0, corners = 0, pt = 0;
        for (uint32_t v0 = 0; v0 < nverbs; v0 += WAVE) {
            const bool in = v0 + (uint32_t)l < nverbs;
            const uint8_t verb = in ? P.in.verbs[vb + v0 + l] : (uint8_t)LYG_VERB_END;
            const uint32_t np = in ? verb_points(verb) : 0u;
            const uint32_t incl = incl_scan(np);
            const bool opens = in && verb <= LYG_VERB_BEGIN;
            uint32_t cnt = 0, cor = 0;
            bool too_long = false;
            if (opens) {
                VRec r;
                decode_verb(verb, pts, npts, pt + incl - np, o.tolerance, r);
                cnt = r.nA + r.nB;
                cor = r.nB ? 2u : 1u;
                too_long = r.nA > MAX_CURVE_POINTS || r.nB > MAX_CURVE_POINTS;
                if (too_long) cnt = 0;
            }
            const uint64_t om = ballot(opens);
            const bool prev_open = l == 0 ? open : ((om >> (l - 1)) & 1ull) != 0;
            if (ballot(in && (verb == LYG_VERB_BEGIN) == prev_open)) bad = true;
            if (ballot(too_long)) space = true;
            raw += readlane_u(incl_scan(cnt), WAVE - 1);
            corners += readlane_u(incl_scan(cor), WAVE - 1);
            ends += (uint32_t)__builtin_popcountll(ballot(in && !opens));
            pt += readlane_u(incl, WAVE - 1);
            const uint32_t last = min((uint32_t)WAVE, nverbs - v0) - 1u;
            open = ((om >> last) & 1ull) != 0;
        }
        if (open) bad = true;
        if (raw > 0xfffffffeull) raw = 0xffffffffull;
        const bool run = !bad && !space;
        if (l == 0) {
            P.raw_n[path] = run ? (uint32_t)raw : 0u;
            P.win_n[path] = run ? (uint32_t)((raw + WIN - 1) / WIN) : 0u;
            P.tail_n[path] = run ? ends : 0u;
            P.att_cap_n[path] = run ? 2u * corners : 0u;
            P.path_mode[path] = run ? 0u : bad ? 1u : 2u;
            if (raw > P.few) P.ctr[5] = 1u;
            P.path_status[path] = bad || !space ? 0u : (uint32_t)LYG_ERR_NO_SPACE;
        }
    }
}

// Wave per path: windows of 64 flattened points, one per lane; the kept ones are written
// end to end with their running length.  Bound by that length's serial f32 sum (64 dependent
// additions per window); the rest of a window is lane-parallel.  10,000 paths, 81 M points:
// 7.6 ms with the windows' t chains in closed form and the edges with side lines listed through
// one counter for all paths, 2.6 ms with t_table and a list per path.
__global__ void __launch_bounds__(64) vw_points_kernel(VWPar P) {
    using namespace vw;
    __shared__ VRec recs[WAVE];
    __shared__ VX vxs[WAVE];
    __shared__ float ts_tab[T_SPAN / 16];
    const int l = lane_id();
    const float nan = __builtin_nanf("");
    for (uint32_t path = blockIdx.x; path < P.in.n_paths; path += gridDim.x) {
        if (P.path_mode[path] != 0u || P.raw_n[path] == 0u) {
            if (l == 0) P.kept_n[path] = 0;
            continue;
        }
        const lyg_stroke_options o = P.opts[P.opts_stride ? path : 0];
        const float thr = ffmax(ffmin(o.tolerance * o.tolerance * 0.5f,
                                      o.line_width * o.line_width * 0.05f),
                                1e-8f);  // StrokeBuilderImpl::new (stroke.rs:591-631)
        const uint32_t vb = P.in.verb_off[path], nverbs = P.in.verb_off[path + 1] - vb;
        const uint32_t pb = P.in.point_off[path], npts = P.in.point_off[path + 1] - pb;
        const float* pts = P.in.points + 2ull * pb;
        const uint32_t kbase = P.raw_off[path], wbase = P.win_off[path];
        const uint32_t tbase = P.tail_off[path], abase = P.att_off[path];
        const uint32_t acap = P.att_off[path + 1] - abase;
        auto width = [&](uint32_t i) {
            return i < npts ? P.widths[(size_t)(pb + i) * P.widths_stride] : nan;
        };
        // carried from window to window
        uint32_t kept = 0, n_att = 0, n_tail = 0, sub_first = 0, sp_cnt = 0;
        vec2 last = mk(nan, nan), last2 = last;  // the last two kept points
        bool last_flat = false, last_hole = false, dead = false, mnec = false;
        float acc = 0.0f, start_adv = 0.0f;  // running length, StrokeBuilderImpl's sub_path_start
        uint32_t pt = 0;
        for (uint32_t v0 = 0; v0 < nverbs; v0 += WAVE) {
            const uint32_t nch = min((uint32_t)WAVE, nverbs - v0);
            const bool in = (uint32_t)l < nch;
            const uint8_t verb = in ? P.in.verbs[vb + v0 + l] : (uint8_t)LYG_VERB_END;
            const uint32_t np = in ? verb_points(verb) : 0u;
            const uint32_t np_incl = incl_scan(np);
            const uint32_t p = pt + np_incl - np;
            pt += readlane_u(np_incl, WAVE - 1);
            VRec r;
            VX x{0.0f, 0.0f, -1.0f, 0, 0};
            uint32_t cnt = 0;
            if (in) {
                decode_verb(verb, pts, npts, p, o.tolerance, r, &x.ts);
                cnt = r.nA + r.nB;
                const uint32_t e = p + (np ? np - 1u : 0u);  // the verb's endpoint
                x.w1 = o.line_width * width(e);
                x.id1 = pb + e;
                if (verb == LYG_VERB_QUADRATIC || verb == LYG_VERB_CUBIC) {
                    x.w0 = o.line_width * width(p - 1u);
                    x.id0 = pb + p - 1u;
                }
            }
            const uint32_t cnt_incl = incl_scan(cnt);
            r.off = cnt_incl - cnt;
            const uint32_t nsteps = readlane_u(cnt_incl, WAVE - 1);
            wave_sync();
            if (in) {
                recs[l] = r;
                vxs[l] = x;
            }
            wave_sync();
            for (uint32_t w0 = 0; w0 < nsteps; w0 += WAVE) {
                const uint32_t t0_step = w0 & ~(T_SPAN - 1u);
                if (w0 == t0_step) {
                    wave_sync();
                    t_table(ts_tab, r, in, w0, nsteps);
                    wave_sync();
                }
                const uint32_t g = w0 + (uint32_t)l;
                const bool valid = g < nsteps;
                vec2 pos = mk(nan, nan);
                float hw = 0.0f, tw = 1.0f;
                uint32_t id0 = 0, id1 = 0;
                bool isB = false, isE = false, close = false, flat = false;
                if (valid) {
                    int lo = 0, hi = (int)nch - 1;  // last verb whose offset <= g
                    while (lo < hi) {
                        const int mid = (lo + hi + 1) >> 1;
                        if (recs[mid].off <= g) lo = mid;
                        else hi = mid - 1;
                    }
                    const VRec& vr = recs[lo];
                    const VX& vx = vxs[lo];
                    const uint32_t k = g - vr.off;
                    const uint32_t kind = vr.kind & 0xffu;
                    id0 = id1 = vx.id1;
                    if (kind == K_END) {
                        isE = true;
                        close = (vr.kind >> 8) != 0;
                    } else if (kind == K_BEGIN || kind == K_LINE) {
                        isB = kind == K_BEGIN;
                        pos = vr.toA;
                        hw = vx.w1 * 0.5f;
                    } else {  // curve_piece
                        const bool cubic = kind == K_CUBIC;
                        const bool inA = k < vr.nA;
                        const uint32_t j = (inA ? k : k - vr.nA) + 1u;
                        float t1 = 1.0f;
                        if (j == (inA ? vr.nA : vr.nB)) {
                            pos = inA ? vr.toA : vr.toB;
                        } else {
                            t1 = t_at(ts_tab, t0_step, g, j, inA ? vr.sA : vr.sB);
                            pos = horner(vr, !inA, inA && cubic, t1);
                        }
                        const bool split = !cubic && vx.ts > 0.0f;
                        const float t0 = split && !inA ? vx.ts : 0.0f;
                        const float ts = split ? (inA ? vx.ts : 1.0f - vx.ts) : 1.0f;
                        tw = ts == 1.0f && t0 == 0.0f ? t1 : t0 + t1 * ts;
                        hw = (vx.w0 * (1.0f - tw) + vx.w1 * tw) * 0.5f;
                        flat = t1 != 1.0f;
                        if (tw != 1.0f) id0 = vx.id0;
                    }
                }
                const uint64_t validm = ballot(valid), begm = ballot(isB), endm = ballot(isE);
                const int nvalid = __builtin_popcountll(validm);
                // ---- which points are kept (stroke.rs:1382-1391) ----
                vec2 rp = shfl_v(pos, l > 0 ? l - 1 : 0);
                if (l == 0) rp = last;
                uint64_t keptm = validm & ~endm;
                bool my_mnec;
                if (ballot(valid && !isE && !isB && sqlen(sub(rp, pos)) < thr) == 0ull) {
                    my_mnec = (begm & mask_le(l)) ? false : mnec;
                } else {
                    vec2 lk = last;
                    uint32_t ck = sp_cnt;
                    bool mn = mnec;
                    my_mnec = false;
                    for (int i = 0; i < nvalid; ++i) {
                        const vec2 pi = readlane_v(pos, i);
                        if ((endm >> i) & 1ull) {
                            ck = 0;
                        } else if ((begm >> i) & 1ull) {
                            mn = false;
                            ck = 1;
                            lk = pi;
                        } else if (sqlen(sub(lk, pi)) < thr) {
                            if (ck == 1) mn = true;
                            keptm &= ~(1ull << i);
                        } else {
                            ck += 1;
                            lk = pi;
                        }
                        if (l == i) my_mnec = mn;
                    }
                }
                const bool kp = (keptm >> l) & 1ull;
                const uint64_t below = keptm & mask_lt(l);
                const uint32_t kidx = kept + (uint32_t)__builtin_popcountll(below);
                // the kept point before, and the one before it
                const int pl = highest_bit(below);
                const int plc = pl < 0 ? 0 : pl;
                vec2 prev = shfl_v(pos, plc);
                bool pflat = shfl_u(flat ? 1u : 0u, plc) != 0;
                if (pl < 0) {
                    prev = last;
                    pflat = last_flat;
                }
                vec2 prev2 = shfl_v(prev, plc);
                if (pl < 0) prev2 = last2;
                const bool inner = kp && !isB;  // has an edge to it
                const bool fastp = pflat && dot(sub(prev, prev2), sub(pos, prev)) > 0.0f;
                const bool hole = inner && pflat && flat && !fastp;
                bool phole = shfl_u(hole ? 1u : 0u, plc) != 0;
                if (pl < 0) phole = last_hole;
                // two joins in a row without side lines or fast path: no length from here on
                const uint64_t deadm = ballot(inner && phole && !fastp);
                const float d = inner ? vlen(sub(pos, prev)) : 0.0f;
                float adv = 0.0f;
                if ((begm | endm) == 0ull) {
                    // lane i adds the lengths up to its own, all lanes in step (a dropped
                    // point adds 0, which leaves the sum as it is)
                    float a = acc;
#pragma unroll
                    for (int i = 0; i < WAVE; ++i) {
                        const float di = readlane_f(d, i);
                        a = a + (l >= i ? di : 0.0f);
                    }
                    adv = dead || (deadm & mask_le(l)) ? nan : a;
                    acc = readlane_f(a, WAVE - 1);
                    dead = dead || deadm != 0ull;
                } else {
                    uint32_t sf = sub_first;
                    for (int i = 0; i < nvalid; ++i) {
                        if ((endm >> i) & 1ull) {
                            const uint32_t m = readlane_u(kidx, i) - sf;
                            const bool cl = (ballot(close) >> i) & 1ull;
                            // end_with_caps sets it from the last edge (stroke.rs:1350)
                            if (m >= 2 && !(cl && m > 2)) start_adv = dead ? nan : acc;
                        } else if ((begm >> i) & 1ull) {
                            acc = start_adv;
                            dead = false;
                            sf = readlane_u(kidx, i);
                        } else if ((keptm >> i) & 1ull) {
                            acc = acc + readlane_f(d, i);
                            dead = dead || ((deadm >> i) & 1ull);
                        }
                        if (l == i) adv = dead ? nan : acc;
                    }
                }
                const bool att = inner && (!pflat || !flat);
                const uint64_t attm = ballot(att);
                const uint32_t ord = n_att + (uint32_t)__builtin_popcountll(attm & mask_lt(l));
                if (kp) {
                    const uint32_t slot = kbase + kidx;
                    reinterpret_cast<float4*>(P.rec)[slot] = make_float4(pos.x, pos.y, hw, adv);
                    P.pflags[slot] = (uint8_t)((flat ? PF_FLAT : 0u) | (isB ? PF_FIRST : 0u) |
                                               (att ? PF_ATT : 0u));
                    if (P.src_t) {
                        P.src_t[slot] = tw;
                        P.src_id[2ull * slot] = id0;
                        P.src_id[2ull * slot + 1] = id1;
                    }
                    if (kidx % WIN == 0u) P.win_att[wbase + kidx / WIN] = ord;
                }
                if (attm) {
                    const uint32_t tot = (uint32_t)__builtin_popcountll(attm);
                    if (n_att + tot > acap) {  // cannot happen: a curve's last point only
                        if (l == 0) mark_slow(P, path);
                    } else if (att) {
                        P.att_point[abase + ord] = kbase + kidx;
                    }
                    n_att += tot;
                }
                if (isE) {
                    const int bl = highest_bit(begm & mask_lt(l));
                    const uint32_t f =
                        bl < 0 ? sub_first
                               : kept + (uint32_t)__builtin_popcountll(keptm & mask_lt(bl));
                    VWTail t{};
                    t.path = path;
                    t.first = f;
                    t.count = kidx - f;
                    t.flags = (close ? 1u : 0u) | (my_mnec ? 2u : 0u);
                    P.tails[tbase + n_tail + (uint32_t)__builtin_popcountll(endm & mask_lt(l))] = t;
                }
                // ---- carry ----
                const int hb = highest_bit(begm), he = highest_bit(endm);
                if (hb >= 0)
                    sub_first = kept + (uint32_t)__builtin_popcountll(keptm & mask_lt(hb));
                if (he >= 0 && he > hb) sp_cnt = 0;
                else if (hb >= 0)
                    sp_cnt = (uint32_t)__builtin_popcountll(keptm & ~mask_lt(hb));
                else sp_cnt += (uint32_t)__builtin_popcountll(keptm);
                n_tail += (uint32_t)__builtin_popcountll(endm);
                mnec = readlane_u(my_mnec ? 1u : 0u, nvalid - 1) != 0;
                const int hk = highest_bit(keptm);
                if (hk >= 0) {
                    last2 = readlane_v(prev, hk);
                    last = readlane_v(pos, hk);
                    last_flat = readlane_u(flat ? 1u : 0u, hk) != 0;
                    last_hole = readlane_u(hole ? 1u : 0u, hk) != 0;
                }
                kept += (uint32_t)__builtin_popcountll(keptm);
            }
        }
        if (l == 0) P.kept_n[path] = kept;
    }
}

// Lane per slot of an edge with an endpoint at one end: the normals of its two side lines (attachments).
__global__ void __launch_bounds__(256) vw_att_kernel(VWPar P) {
    const uint32_t n = P.att_off[P.in.n_paths];
    const float PI = 3.14159265358979323846f;
    for (uint32_t slot = blockIdx.x * 256u + threadIdx.x; slot < n; slot += gridDim.x * 256u) {
        const uint32_t i = P.att_point[slot];
        if (i == 0xffffffffu) continue;
        const float4 p0 = reinterpret_cast<const float4*>(P.rec)[i - 1];
        const float4 p1 = reinterpret_cast<const float4*>(P.rec)[i];
        const vec2 e = sub(mk(p1.x, p1.y), mk(p0.x, p0.y));
        const float d = vlen(e);
        const float ea = angle_of(e);
        float va = (float)asin((double)((p1.z - p0.z) / d));
        if (va != va) va = 0.0f;
        const float n0 = ea + 1.0f * (PI * 0.5f + va), n1 = ea + -1.0f * (PI * 0.5f + va);
        reinterpret_cast<float4*>(P.att_n)[slot] =
            make_float4(t_cos(n0), t_sin(n0), t_cos(n1), t_sin(n1));
    }
}

// Wave per window of 63 joins.  EMIT false: the window's vertices and triangles, and the
// joins that may fold back.  EMIT true: the geometry at the scanned offsets, the ids the
// sub-paths' ends need.  List: the windows of `dirty` only (counted again).
template <bool EMIT>
__global__ void __launch_bounds__(256) vw_window_kernel(VWPar P, uint32_t list, uint32_t chunk) {
    using namespace vw;
    __shared__ ArcJob jobs_all[EMIT ? 4 : 1][EMIT ? 2 * WAVE : 1];
    __shared__ uint32_t ax_all[EMIT ? 4 : 1][EMIT ? WAVE : 1], ac_all[EMIT ? 4 : 1][EMIT ? WAVE : 1];
    const int l = lane_id();
    const int wv = EMIT ? (int)(threadIdx.x / WAVE) : 0;
    const uint32_t wave = blockIdx.x * 4u + threadIdx.x / WAVE, n_waves = gridDim.x * 4u;
    const uint32_t n_win = list ? min(P.ctr[3], P.dirty_cap) : P.n_windows;
    for (uint32_t c0 = wave * chunk; c0 < n_win; c0 += n_waves * chunk) {
        uint32_t path = 0, wend = 0;  // the path of the windows before `wend`
        bool run = false;
        PC c;
        const uint32_t c1 = min(n_win, c0 + chunk);
        // EMIT: where the next window has to start, and whether one did not
        uint32_t next_v = EMIT ? P.win_voff[c0] : 0u, next_t = EMIT ? P.win_ioff[c0] : 0u;
        uint32_t differ = 0;
        for (uint32_t k = c0; k < c1; ++k) {
            const uint32_t w = list ? P.dirty[k] : k;
            if (w >= wend || list) {
                path = wave_search_last_le(P.win_off, P.in.n_paths + 1u, w);
                wend = P.win_off[path + 1];
                run = P.path_mode[path] == 0u;
                if (run) c = path_ctx(P, path);
            }
            const uint32_t wb = P.win_off[path];
            const uint32_t start = (w - wb) * WIN;
            if (!run || start >= c.kn) {
                if (!EMIT && l == 0) P.win_nv[w] = P.win_ni[w] = 0u;
                if (EMIT && !run) {  // a path left to the serial kernel after it was counted
                    next_v = P.win_voff[w + 1u];
                    next_t = P.win_ioff[w + 1u];
                }
                continue;
            }
            uint32_t i = start + (uint32_t)l - 1u, back = 0;
            bool valid = l > 0 && i < c.kn;
            uint32_t f = valid ? c.fl[i] : 0u;
            if (l == 0 && start > 0u) {  // the last buffered point before the window
                valid = true;
                f = c.fl[i];
                while (f & PF_SKIP) {
                    back += (f & PF_ATT) ? 1u : 0u;
                    f = c.fl[--i];
                }
                back += (f & PF_ATT) ? 1u : 0u;
            }
            const uint64_t attm = ballot(valid && l > 0 && (f & PF_ATT));
            const uint32_t watt = P.win_att[w];
            const uint32_t ord =
                l == 0 ? watt - back : watt + (uint32_t)__builtin_popcountll(attm & mask_lt(l));
            const bool last = valid && (i + 1u >= c.kn || (c.fl[i + 1u] & PF_FIRST));
            const bool isj = valid && !last && !(f & (PF_FIRST | PF_SKIP));
            JInfo J;
            uint32_t q = 0;
            bool pfirst = false;
            uint32_t code = LC_FIRST;
            if (isj) {
                join_at(c, i, ord, J, q, pfirst);
                code = join_code(J);
            }
            const uint64_t bufm = ballot(valid && !(f & PF_SKIP));
            const int lq = highest_bit(bufm & mask_lt(l));
            const uint32_t pcode = shfl_u(code, lq < 0 ? 0 : lq);
            uint32_t nv = 0, nt = 0;
            if (isj) join_counts(J, pcode, !pfirst && l > 0, &nv, &nt);
            const uint32_t nv0 = readlane_u(nv, 0);
            if (!EMIT) {
                if (l == 0) nv = nt = 0;
                const uint32_t tv = readlane_u(incl_scan(nv), WAVE - 1);
                const uint32_t tt = readlane_u(incl_scan(nt), WAVE - 1);
                if (l == 0) {
                    P.win_nv[w] = tv;
                    P.win_ni[w] = tt;
                }
                if (!list && isj && l > 0 && J.weird) {
                    P.pflags[P.raw_off[path] + i] = (uint8_t)(f | PF_CAND);
                    const uint32_t s = atomicAdd(&P.ctr[2], 1u);
                    if (s < P.cand_cap) {
                        P.cands[2ull * s] = path;
                        P.cands[2ull * s + 1] = i;
                    } else {
                        atomicOr(&P.ctr[4], 1u);
                    }
                }
                continue;
            }
            VWTail* tail = nullptr;
            if (l > 0 && (last || (isj && pfirst))) tail = tail_of(P, path, i);
            if (l == 0) nv = nt = 0;
            if (last) {
                nv = l > 0 ? tail->nv : 0u;
                nt = l > 0 ? tail->nt : 0u;
            }
            const uint32_t w_v = P.win_voff[w], w_t = P.win_ioff[w];
            const uint32_t v_at = w_v - P.win_voff[wb];
            const uint32_t t_at = w_t - P.win_ioff[wb];
            differ |= (w_v ^ next_v) | (w_t ^ next_t);
            const uint32_t vi = incl_scan(nv), ti = incl_scan(nt);
            const uint32_t vx = vi - nv, tx = ti - nt;
            next_v = w_v + readlane_u(vi, WAVE - 1);
            next_t = w_t + readlane_u(ti, WAVE - 1);
            const uint32_t my_v = l == 0 ? v_at - nv0 : v_at + vx;
            const uint32_t pv = shfl_u(my_v, lq < 0 ? 0 : lq);
            const uint32_t v0 = P.vtx_off[path], id_base = P.vertex_offset + v0;
            const uint32_t i0 = P.idx_off[path], i1 = P.idx_off[path + 1];
            const uint32_t vlim = P.vtx_off[path + 1] - v0;
            const bool own = isj && l > 0;
            Sink s;
            s.emit = true;
            s.err = P.err;
            s.nv = s.ni = 0;
            s.vid0 = id_base;
            s.vid = id_base + my_v;
            s.vout = P.out_vertices + 2ull * v0;
            s.vlim = vlim;
            const uint32_t at = 3u * (t_at + tx);
            s.iout = P.out_indices + (size_t)i0 + at;
            s.ileft = i1 - i0 > at ? i1 - i0 - at : 0u;
            ArcJobs aj;
            if (own) {
                EPD pe;
                ids_of(pcode, id_base + pv, pe.pv, pe.nv);
                pe.fold[SP] = (pcode & LC_FOLD_P) ? 1 : 0;
                pe.fold[SN] = (pcode & LC_FOLD_N) ? 1 : 0;
                SParams sp{};
                sp.hw = c.rec[i].z;
                join_emit(J, pe, !pfirst, sp, s, &aj);
                if (pfirst) tail->f1_base = my_v;
            }
            if (tail && last) {
                tail->p_base = pv;
                tail->v_at = my_v;
                tail->t_at = t_at + tx;
            }
            emit_arcs<true>(aj, s, 0.0f, jobs_all[wv], ax_all[wv], ac_all[wv]);
            if (P.out_attrs && own) {
                const size_t slot = P.raw_off[path] + (size_t)i;
                const float t = P.src_t[slot];
                const float* a = P.attrs + (size_t)P.src_id[2 * slot] * P.n_attrs;
                const float* b = P.attrs + (size_t)P.src_id[2 * slot + 1] * P.n_attrs;
                const bool edge = t != 1.0f;
                for (uint32_t v = my_v; v < my_v + nv && v < vlim; ++v) {
                    float* d = P.out_attrs + ((size_t)v0 + v) * P.n_attrs;
                    for (uint32_t x = 0; x < P.n_attrs; ++x)
                        d[x] = edge ? a[x] * (1.0f - t) + b[x] * t : a[x];
                }
            }
        }
        // the count saw other joins than these
        if (EMIT && (differ | (P.win_voff[c1] ^ next_v) | (P.win_ioff[c1] ^ next_t)) != 0u && l == 0)
            atomicOr(P.err, 4u);
    }
}

// A candidate that is the first of its group: none in the 8 points before it on its curve.
__device__ __forceinline__ bool skip_leader(const uint8_t* fl, uint32_t i) {
    for (uint32_t b = 1; b <= 8u && b <= i && (fl[i - b] & vw::PF_FLAT); ++b)
        if (fl[i - b] & vw::PF_CAND) return false;
    return true;
}

// Thread per candidate of the count pass: settles which joins fold back.  A skip only changes
// what the next points see before them, and nothing beyond the curve's end, which is never
// skipped (whether a join after it folds back depends on points from there on).  So the first
// candidate of a group walks on along its curve until 8 joins in a row are neither skipped nor
// candidates.  Skips that the count could not see may bring it to the next group, whose own
// thread has then read flags from before them: the path is left to the serial kernel.
//
// A skip changes the counts of up to four buffered points after it, and past the curve's end
// those of the end's join and of the point after that: all windows of the walk are counted
// again, and that of the two points after a walk to the end.
__global__ void __launch_bounds__(64) vw_skip_kernel(VWPar P) {
    using namespace vw;
    const uint32_t n = min(P.ctr[2], P.cand_cap);
    for (uint32_t k = blockIdx.x * 64u + threadIdx.x; k < n; k += gridDim.x * 64u) {
        const uint32_t path = P.cands[2ull * k], i = P.cands[2ull * k + 1];
        if (P.path_mode[path] != 0u) continue;
        const PC c = path_ctx(P, path);
        uint8_t* fl = P.pflags + P.raw_off[path];
        if (!skip_leader(fl, i)) continue;
        uint32_t clean = 0, x = i;
        for (; clean < 8u && x + 1u < c.kn && (fl[x] & PF_FLAT) && !(fl[x + 1u] & PF_FIRST); ++x) {
            const bool cand = (fl[x] & PF_CAND) != 0;
            if (cand && x != i && skip_leader(fl, x)) {
                mark_slow(P, path);
                break;
            }
            JInfo J;
            uint32_t q;
            bool pfirst;
            join_at(c, x, att_ord(c, x), J, q, pfirst);
            if (q + 1u != x && (fl[x + 1u] & PF_FLAT)) {
                // the running lengths were written as if the point before had stayed
                const vec2 a = pos_of(c.rec[x - 1u]), j = pos_of(c.rec[x]);
                const bool naive = dot(sub(j, a), sub(pos_of(c.rec[x + 1u]), j)) > 0.0f;
                if (naive != J.fast) mark_slow(P, path);
            }
            clean = cand || J.weird ? 0u : clean + 1u;
            if (J.weird) fl[x] = (uint8_t)(fl[x] | PF_SKIP);
        }
        const uint32_t last = min(x + 2u, c.kn - 1u);
        for (uint32_t w = i / WIN; w <= last / WIN; ++w) {
            const uint32_t s = atomicAdd(&P.ctr[3], 1u);
            if (s < P.dirty_cap) P.dirty[s] = P.win_off[path] + w;
            else atomicOr(&P.ctr[4], 1u);
        }
    }
}

// Lane per sub-path: its end (end_sub), from the states of its first two and last two
// buffered points.  Counting adds to the window of the sub-path's last point.
template <bool EMIT>
__global__ void __launch_bounds__(64) vw_tail_kernel(VWPar P) {
    using namespace vw;
    for (uint32_t k = blockIdx.x * 64u + threadIdx.x; k < P.n_tails; k += gridDim.x * 64u) {
        VWTail& t = P.tails[k];
        const uint32_t path = t.path;
        if (P.path_mode[path] != 0u) continue;
        const lyg_stroke_options o = P.opts[P.opts_stride ? path : 0];
        const PC c = path_ctx(P, path);
        const size_t slot0 = P.raw_off[path];
        const uint32_t first = t.first, L = t.first + t.count - 1u;
        Sink sk;
        sk.nv = sk.ni = 0;
        sk.emit = EMIT;
        sk.err = EMIT ? P.err : nullptr;
        const uint32_t id_base = EMIT ? P.vertex_offset + P.vtx_off[path] : 0u;
        if (EMIT) {
            const uint32_t n_i = P.idx_off[path + 1] - P.idx_off[path];
            sk.vid0 = id_base;
            sk.vid = id_base + t.v_at;
            sk.vout = P.out_vertices + 2ull * P.vtx_off[path];
            sk.vlim = P.vtx_off[path + 1] - P.vtx_off[path];
            sk.iout = P.out_indices + (size_t)P.idx_off[path] + 3u * t.t_at;
            sk.ileft = n_i > 3u * t.t_at ? n_i - 3u * t.t_at : 0u;
        } else {
            // ids are only compared: the new ones start above the stand-ins of the joins
            sk.vid = sk.vid0 = 0x80000000u;
            sk.vout = nullptr;
            sk.iout = nullptr;
            sk.vlim = sk.ileft = 0;
        }
        Stroker S;
        S.lw = o.line_width;
        S.tol = o.tolerance;
        S.miter_limit = o.miter_limit;
        S.merge2 = ffmax(ffmin(o.tolerance * o.tolerance * 0.5f,
                               o.line_width * o.line_width * 0.05f),
                         1e-8f);
        S.start_cap = o.start_cap;
        S.end_cap = o.end_cap;
        S.line_join = o.line_join;
        S.s = &sk;
        S.on_path = mk(0.0f, 0.0f);
        S.vhw = o.line_width * 0.5f;
        S.count = 0;
        S.n_firsts = 0;
        S.may_need_empty_cap = (t.flags & 2u) != 0;
        S.sub_path_start_adv = 0.0f;
        S.status = 0;
        S.attrs = P.attrs;
        S.n_attrs = P.n_attrs;
        S.attr_out = EMIT && P.out_attrs ? P.out_attrs + (size_t)P.vtx_off[path] * P.n_attrs
                                         : nullptr;
        S.sf = S.sto = 0;
        S.st = 0.0f;
        S.sedge = false;
        S.filled = sk.vid;
        // a point as step() buffers it, before its join
        auto point = [&](Pt& e, uint32_t i) {
            const float4 r = c.rec[i];
            pt_init(e, mk(r.x, r.y), r.z, c.join, (c.fl[i] & PF_FLAT) != 0);
            e.adv = r.w;
            if (i > first && (c.fl[i] & PF_FLAT) && (c.fl[i - 1u] & PF_FLAT) && !fast_at(c, i - 1u))
                e.adv = __builtin_nanf("");
            if (S.attr_out) {
                const size_t s = slot0 + i;
                e.st = P.src_t[s];
                e.sf = P.src_id[2 * s];
                e.sto = P.src_id[2 * s + 1];
                e.sedge = e.st != 1.0f;
            }
        };
        // its side points towards the next point
        auto next_sides = [&](Pt& e, uint32_t i) {
            if (!(c.fl[i + 1u] & PF_ATT)) return;
            const float4 a = c.att[att_ord(c, i + 1u)];
            e.sp[SP].next = add(e.pos, mul(mk(a.x, a.y), e.hw));
            e.sp[SN].next = add(e.pos, mul(mk(a.z, a.w), e.hw));
        };
        // after its join
        auto joined = [&](Pt& e, uint32_t i, uint32_t base) {
            point(e, i);
            JInfo J;
            uint32_t q;
            bool pfirst;
            join_at(c, i, att_ord(c, i), J, q, pfirst);
            // a fast join fills a missing running length in; it was written filled
            if (J.fast) e.adv = c.rec[i].w;
            ids_of(join_code(J), base, J.x.pv, J.x.nv);
#pragma unroll
            for (int k2 = 0; k2 < 2; ++k2) {
                e.sp[k2].prev = J.x.prev[k2];
                e.sp[k2].next = J.x.next[k2];
                e.sp[k2].single = J.x.single[k2];
                e.sp[k2].has_single = J.x.has_single[k2] != 0;
                e.sp[k2].prev_v = J.x.pv[k2];
                e.sp[k2].next_v = J.x.nv[k2];
                e.fold[k2] = J.x.fold[k2] != 0;
            }
            e.join = J.x.line_join;
        };
        Pt pl;
        point(pl, L);
        if (t.count == 1u) {
            S.buf[0] = pl;
            S.count = 1;
        } else {
            if (c.fl[L] & PF_ATT) {
                const float4 a = c.att[att_ord(c, L)];
                pl.sp[SP].prev = add(pl.pos, mul(mk(a.x, a.y), pl.hw));
                pl.sp[SN].prev = add(pl.pos, mul(mk(a.z, a.w), pl.hw));
            }
            const uint32_t q = eff_prev(c, L);
            Pt p0;
            point(p0, first);
            next_sides(p0, first);
            if (q == first) {
                S.buf[0] = p0;
                S.buf[1] = pl;
                S.count = 2;
            } else {
                uint32_t f1 = first + 1u;
                while (c.fl[f1] & PF_SKIP) ++f1;
                S.firsts[0] = p0;
                joined(S.firsts[1], f1, EMIT ? id_base + t.f1_base : 8u * (f1 - first));
                S.n_firsts = 2;
                joined(S.buf[1], q, EMIT ? id_base + t.p_base : 8u * (q - first));
                S.buf[0] = S.buf[1];  // the oldest buffered point is not read again
                S.buf[2] = pl;
                S.count = 3;
            }
        }
        end_sub(S, (t.flags & 1u) != 0);
        flush_attrs(S);
        if (!EMIT) {
            t.nv = sk.nv;
            t.nt = sk.ni;
            const uint32_t w = P.win_off[path] + L / WIN;
            if (sk.nv) atomicAdd(&P.win_nv[w], sk.nv);
            if (sk.ni) atomicAdd(&P.win_ni[w], sk.ni);
        }
    }
}

// Per path: its counts from its windows' offsets, or its place in the list of those that the
// serial kernel counts (a counter's addition per wave: one per path took 360 us of 30,000).
__global__ void __launch_bounds__(256) vw_totals_kernel(VWPar P) {
    const uint32_t n = P.in.n_paths;
    for (uint32_t p0 = blockIdx.x * 256u; p0 < n; p0 += gridDim.x * 256u) {
        const uint32_t p = p0 + threadIdx.x;
        const bool serial = p < n && P.path_mode[p] == 1u;
        const uint64_t m = ballot(serial);
        if (m) {
            const uint32_t at =
                readlane_u(atomicAdd(&P.ctr[1], lane_id() == 0 ? (uint32_t)__popcll(m) : 0u), 0);
            if (serial) P.slow_list[at + (uint32_t)__popcll(m & mask_lt(lane_id()))] = p;
        }
        if (p >= n || serial) continue;
        const uint32_t a = P.win_off[p], b = P.win_off[p + 1];
        P.path_nv[p] = P.win_voff[b] - P.win_voff[a];
        P.path_ni[p] = 3u * (P.win_ioff[b] - P.win_ioff[a]);
    }
}

}  // namespace lyg

extern "C" {

hipError_t lyg_launch_stroke_vw(const lyg::StrokeVWLaunch* L, int emit, int grid,
                                hipStream_t s) {
    if (L->in.n_paths == 0) return hipSuccess;
    if (emit)
        hipLaunchKernelGGL(lyg::stroke_vw_kernel<true>, dim3(grid), dim3(64), 0, s, *L);
    else
        hipLaunchKernelGGL(lyg::stroke_vw_kernel<false>, dim3(grid), dim3(64), 0, s, *L);
    return hipGetLastError();
}


hipError_t lyg_launch_vw_plan(const lyg::VWPar* P, int grid, hipStream_t s) {
    hipLaunchKernelGGL(lyg::vw_plan_kernel, dim3(grid), dim3(64), 0, s, *P);
    return hipGetLastError();
}
// The kept points, the side lines, the windows' and sub-paths' counts, the per-path totals'
// inputs (the windows' scans and vw_totals follow).
hipError_t lyg_launch_vw_count(const lyg::VWPar* P, int grid_paths, int grid_win, uint32_t chunk,
                               hipStream_t s) {
    hipLaunchKernelGGL(lyg::vw_points_kernel, dim3(grid_paths), dim3(64), 0, s, *P);
    hipLaunchKernelGGL(lyg::vw_att_kernel, dim3(grid_win), dim3(256), 0, s, *P);
    hipLaunchKernelGGL(lyg::vw_window_kernel<false>, dim3(grid_win), dim3(256), 0, s, *P, 0u, chunk);
    hipLaunchKernelGGL(lyg::vw_skip_kernel, dim3(16), dim3(64), 0, s, *P);
    hipLaunchKernelGGL(lyg::vw_window_kernel<false>, dim3(16), dim3(256), 0, s, *P, 1u, 1u);
    if (P->n_tails)
        hipLaunchKernelGGL(lyg::vw_tail_kernel<false>, dim3((P->n_tails + 63) / 64), dim3(64), 0,
                           s, *P);
    return hipGetLastError();
}
hipError_t lyg_launch_vw_totals(const lyg::VWPar* P, hipStream_t s) {
    hipLaunchKernelGGL(lyg::vw_totals_kernel, dim3((P->in.n_paths + 255) / 256), dim3(256), 0, s,
                       *P);
    return hipGetLastError();
}
hipError_t lyg_launch_vw_emit(const lyg::VWPar* P, int grid_win, uint32_t chunk, hipStream_t s) {
    hipLaunchKernelGGL(lyg::vw_window_kernel<true>, dim3(grid_win), dim3(256), 0, s, *P, 0u, chunk);
    if (P->n_tails)
        hipLaunchKernelGGL(lyg::vw_tail_kernel<true>, dim3((P->n_tails + 63) / 64), dim3(64), 0, s,
                           *P);
    return hipGetLastError();
}

}  // extern "C"
