// lyon_algorithms' path validators for gfx950, over the batched path layout:
//
//   * winding numbers / hit tests of query points (path_winding_number_at_position and
//     hit_test_path, crates/algorithms/src/hit_test.rs:8-117): a wave per query point or few.
//     The lanes take the path's verbs 64 at a time; a DPP scan of the points each verb
//     consumes gives every lane its verb's points, a running maximum gives the latest
//     Begin (the sub-path's first point, which End and Close connect back to).  Curves whose
//     place decides their count are not flattened; the others are queued and a lane walks
//     the flattened points of each, counting the crossings left of the query; the count is
//     an integer, so the sum is exact in any order.
//   * approximate signed areas (approximate_signed_area, crates/algorithms/src/area.rs:7-54):
//     lyon's serial f32 sum of cross products in event order; one wave per path computes up to
//     1,024 terms at once and adds them in order, the running value going from lane to lane.
//
// Paths are as lyon's builders make them: every sub-path opens with Begin, so the current
// point of a verb is the last point consumed before it (path.rs:843-909).  Curves are
// flattened as for_each_flattened / Flattened do (quadratic_bezier.rs:337-359, 975-1031;
// cubic_bezier.rs:563-582, 1405-1454): t = step, step + step, ..., the last point `to`.
#include <hip/hip_runtime.h>

#include "lyg_math.h"
#include "lyg_types.h"
#include "wave.h"

namespace lyg {

namespace {

constexpr int VAL_WAVES = 4;

// Points each verb consumes (path.rs:29-36): Line 1, Quadratic 2, Cubic 3, Begin 1,
// Close 1 (the stored first point), End 0.
__device__ __forceinline__ uint32_t points_of(uint32_t verb) {
    return verb < 5u ? (verb == 2u ? 3u : verb == 1u ? 2u : 1u) : 0u;
}

// One path's points; reading past them gives NaN, as PointIter::next does.
struct PathPts {
    const float* p;
    uint32_t n;
    __device__ __forceinline__ vec2 at(uint32_t i) const {
        if (i < n) return mk(p[2ull * i], p[2ull * i + 1]);
        return mk(__builtin_nanf(""), __builtin_nanf(""));
    }
};

// hit_test.rs:85-117 test_segment; LineSegment::sample is euclid's lerp.
__device__ __forceinline__ int seg_winding(vec2 P, vec2 a, vec2 b) {
    const float min_y = ffmin(a.y, b.y), max_y = ffmax(a.y, b.y);
    if (min_y > P.y || max_y <= P.y || ffmin(a.x, b.x) > P.x) return 0;
    if (a.y == b.y) return 0;
    const float d = b.y - a.y;
    const float t = (P.y - a.y) / d;
    const float x = lerp(a, b, t).x;
    if (x > P.x) return 0;
    return d > 0.0f ? 1 : -1;
}

// What is certain about a curve's crossings left of a query without its flattened points.
enum : int { CURVE_NONE, CURVE_LEFT, CURVE_WALK, CURVE_WALK_WHOLE };

// CURVE_NONE: the curve's y range (fast_bounding_range_y, quadratic_bezier.rs:561-566,
// cubic_bezier.rs:906-920) misses P, or every flattened point lies right of P.  CURVE_LEFT:
// they all lie left of it; then each flattened edge counts +1, -1 or 0 by its ends' sides of
// P.y alone and the sum telescopes to the curve's own ends.  The points lie within the
// control points' x range widened by what rounding adds: up to ~60 half ulps of the largest
// coordinate M from the polynomial's terms (|a1|, |a2|, |a3| <= 12 M, five roundings each),
// and t past 1 by at most n half ulps, n the segment count: with (ext_x + ext_y) <= 1e8 tol
// Wang's n is below 17,500 and t below 1.0011, another 0.0034 ext_x.  Both margins are taken
// at least twice.  (A tolerance below 1e-12 could underflow in Wang's formula.)  Anything not finite compares false and is walked whole.
__device__ __forceinline__ int curve_side(vec2 P, uint32_t verb, vec2 f, vec2 c1, vec2 c2,
                                          vec2 to, float tol) {
    const vec2 c = verb == 2u ? c2 : to;
    const float lo = ffmin(ffmin(ffmin(f.y, c1.y), c.y), to.y);
    const float hi = ffmax(ffmax(ffmax(f.y, c1.y), c.y), to.y);
    if (lo > P.y || hi < P.y) return CURVE_NONE;
    const float x0 = ffmin(ffmin(f.x, c1.x), ffmin(c.x, to.x));
    const float x1 = ffmax(ffmax(f.x, c1.x), ffmax(c.x, to.x));
    const float big = ffmax(ffabs(x0), ffabs(x1));
    const float ext = x1 - x0;
    const float margin = 0.01f * ext + 2e-5f * big;
    // sums, so that a NaN coordinate (which the minima pass over) shows
    const float all = (f.x + c1.x + c.x + to.x) + (f.y + c1.y + c.y + to.y);
    const bool sure = ext + (hi - lo) <= 1e8f * tol && tol >= 1e-12f && ffabs(all) <= 1e30f && big <= 1e30f &&
                      ffmax(ffabs(lo), ffabs(hi)) <= 1e30f && P.y == P.y;
    if (sure && x0 - margin > P.x) return CURVE_NONE;
    if (sure && x1 + margin < P.x) return CURVE_LEFT;
    return sure ? CURVE_WALK : CURVE_WALK_WHOLE;
}

// Sum of seg_winding over the flattened edges of a quadratic (verb 1, whose end is `to`) or
// cubic (verb 2), in blocks of 8 edges (more beyond 512: at most 64 blocks).  A first pass
// over the blocks' ends tells most of them apart as curve_side does the curve; the second
// walks the flattened points of the others in lyon's order, t by lyon's serial sum.  A block's
// points lie within its ends' box widened by
//   * the chord's distance, at most |c''| dt^2 / 8 a coordinate: Wang's count makes that the
//     tolerance for dt = 1 / n, and a block spans at most (B + 1) / n (n need not be whole);
//   * what rounding adds (curve_side), t's drift now with the count itself: n half ulps,
//     3 ext per unit of t;
// both rounded up.  Curves that curve_side does not trust are walked whole.
__device__ __forceinline__ int curve_winding(vec2 P, uint32_t verb, vec2 from, vec2 c1, vec2 c2,
                                             vec2 to, bool sure, float tol) {
    const bool cubic = verb == 2u;
    vec2 a1, a2, a3 = mk(0.0f, 0.0f);
    float n;
    if (cubic) {
        n = cubic_wang(from, c1, c2, to, tol);
        a1 = mul(sub(c1, from), 3.0f);
        a2 = add(sub(mul(from, 3.0f), mul(c1, 6.0f)), mul(c2, 3.0f));
        a3 = add(sub(to, from), mul(sub(c1, c2), 3.0f));
    } else {
        n = quad_wang(from, c1, to, tol);
        a1 = mul(sub(c1, from), 2.0f);
        a2 = sub(add(from, to), mul(c1, 2.0f));
    }
    const float step = 1.0f / n;
    const uint32_t cnt = seg_count(n);
    auto point = [&](float t) {
        vec2 v = from;
        float tt = t;
        v = add(v, mul(a1, tt));
        tt = tt * t;
        v = add(v, mul(a2, tt));
        tt = tt * t;
        const vec2 v3 = add(v, mul(a3, tt));
        return cubic ? v3 : v;
    };
    const uint32_t B = cnt <= 512u ? 8u : (cnt + 63u) / 64u;
    const uint32_t nb = (cnt - 1u) / B + 1u;
    uint64_t open = nb >= 64u ? ~0ull : (1ull << nb) - 1ull;
    int w = 0;
    if (sure) {
        const vec2 c = cubic ? c2 : to;
        const float x0 = ffmin(ffmin(from.x, c1.x), ffmin(c.x, to.x));
        const float x1 = ffmax(ffmax(from.x, c1.x), ffmax(c.x, to.x));
        const float y0 = ffmin(ffmin(from.y, c1.y), ffmin(c.y, to.y));
        const float y1 = ffmax(ffmax(from.y, c1.y), ffmax(c.y, to.y));
        const float big = ffmax(ffmax(ffabs(x0), ffabs(x1)), ffmax(ffabs(y0), ffabs(y1)));
        const float ext = ffmax(x1 - x0, y1 - y0);
        const float m = 1.02f * tol * (float)((B + 1u) * (B + 1u)) + 4e-7f * n * ext + 2e-5f * big;
        vec2 a = from;
        for (uint32_t j = 0; j < nb; ++j) {
            const vec2 v = point((float)((j + 1u) * B) * step);
            const vec2 b = j + 1u == nb ? to : v;
            const bool none = ffmin(a.y, b.y) - m > P.y || ffmax(a.y, b.y) + m < P.y ||
                              ffmin(a.x, b.x) - m > P.x;
            const bool left = ffmax(a.x, b.x) + m < P.x && ffabs(a.y - P.y) > m &&
                              ffabs(b.y - P.y) > m;
            if (none || left) open &= ~(1ull << j);
            if (!none && left) w += (b.y > P.y ? 1 : 0) - (a.y > P.y ? 1 : 0);
            a = b;
        }
    }
    float t = 0.0f;
    uint32_t k = 0;  // t is the sum of k steps
    while (open) {
        const uint32_t first = (uint32_t)__builtin_ctzll(open) * B;
        open &= open - 1ull;
        while (k < first) {
            if (B == 8u) {
#pragma unroll
                for (int q = 0; q < 8; ++q) t = t + step;
                k += 8u;
            } else {
                t = t + step;
                ++k;
            }
        }
        vec2 prev = first ? point(t) : from;
        const uint32_t last = first + B < cnt ? first + B : cnt;
        while (k < last) {
            t = t + step;
            ++k;
            const vec2 p = point(t);
            const vec2 v = k == cnt ? to : p;
            w += seg_winding(P, prev, v);
            prev = v;
        }
    }
    return w;
}

}  // namespace

// Curves that have to be walked, of several queries and windows, until 64 fill the lanes.
struct WalkQueue {
    vec2 from[2 * WAVE], c1[2 * WAVE], c2[2 * WAVE], to[2 * WAVE];
    uint32_t what[2 * WAVE];  // the wave's query | verb << 8 | whole << 16
    int32_t winding[WAVE];    // of the wave's queries
    vec2 pos[WAVE];
};

// A wave takes up to 64 consecutive queries (`per_wave`), one after the other.  VALU
// bound: most of a path's curves need no walk (curve_side), and those that do go through a
// queue, so that all lanes walk one each instead of the few that one window yields.
// 100,000 queries on 10,000 paths of 8-256 segments, 17 curves of 168 edges to walk per
// query: 1,352 us with each window's curves walked where they are found, 564 us through the
// queue, 265 us with the blocks of curve_winding.
__global__ void __launch_bounds__(WAVE* VAL_WAVES) winding_kernel(ValidateLaunch L,
                                                                 uint32_t per_wave) {
    __shared__ WalkQueue queues[VAL_WAVES];
    WalkQueue& Q = queues[threadIdx.x / WAVE];
    const int l = lane_id();
    const uint64_t q0 = (uint64_t)(blockIdx.x * VAL_WAVES + threadIdx.x / WAVE) * per_wave;
    if (q0 >= L.n_queries) return;
    const uint32_t nq = L.n_queries - (uint32_t)q0 < per_wave ? L.n_queries - (uint32_t)q0 : per_wave;
    Q.winding[l] = 0;
    if ((uint32_t)l < nq)
        Q.pos[l] = mk(L.queries[2ull * (q0 + l)], L.queries[2ull * (q0 + l) + 1]);
    wave_sync();
    uint32_t queued = 0;
    auto walk = [&](uint32_t first, uint32_t n) {
        if ((uint32_t)l < n) {
            const uint32_t e = first + (uint32_t)l;
            const uint32_t what = Q.what[e];
            const int w =
                curve_winding(Q.pos[what & 255u], what >> 8 & 255u, Q.from[e], Q.c1[e], Q.c2[e],
                              Q.to[e], (what >> 16) == 0u, L.tolerance);
            if (w) atomicAdd(&Q.winding[what & 255u], w);
        }
        wave_sync();
    };
    for (uint32_t k = 0; k < nq; ++k) {
        const uint32_t pid = readlane_u(L.query_path[q0 + k], 0);
        if (pid >= L.n_paths) continue;
        const vec2 P = readlane_v(Q.pos[k], 0);
        const uint32_t vb = L.verb_off[pid], nv = L.verb_off[pid + 1] - vb;
        const uint32_t pb = L.point_off[pid];
        const PathPts pts{L.points + 2ull * pb, L.point_off[pid + 1] - pb};
        uint32_t pc = 0;   // points consumed by the verbs before this window
        uint32_t beg = 0;  // 1 + point index of the latest Begin so far, 0 before any
        int w = 0;
        for (uint32_t c = 0; c < nv; c += WAVE) {
            const uint32_t i = c + (uint32_t)l;
            const uint32_t verb = i < nv ? (uint32_t)L.verbs[vb + i] : 0xffu;
            const uint32_t cons = points_of(verb);
            const uint32_t incl = incl_scan(cons);
            const uint32_t pi = pc + incl - cons;  // this verb's first point
            uint32_t b = incl_max_u32(verb == 3u ? pi + 1u : 0u);
            b = b > beg ? b : beg;
            int side = CURVE_NONE;
            vec2 from = mk(0.0f, 0.0f), c1 = from, c2 = from, to = from;
            if (verb != 3u && verb != 0xffu) {
                from = pts.at(pi - 1u);
                if (verb == 1u || verb == 2u) {
                    c1 = pts.at(pi);
                    c2 = pts.at(pi + 1u);
                    to = verb == 1u ? c2 : pts.at(pi + 2u);
                    side = curve_side(P, verb, from, c1, c2, to, L.tolerance);
                    if (side == CURVE_LEFT) w += (to.y > P.y ? 1 : 0) - (from.y > P.y ? 1 : 0);
                } else {
                    // a line, or End / Close: the edge from the current point to the first
                    w += seg_winding(P, from, verb == 0u ? pts.at(pi) : pts.at(b - 1u));
                }
            }
            const uint64_t walked = ballot(side >= CURVE_WALK);
            if (side >= CURVE_WALK) {
                const uint32_t e = queued + (uint32_t)__builtin_popcountll(walked & mask_lt(l));
                Q.from[e] = from;
                Q.c1[e] = c1;
                Q.c2[e] = c2;
                Q.to[e] = to;
                Q.what[e] = k | verb << 8 | (side == CURVE_WALK ? 0u : 1u << 16);
            }
            queued += (uint32_t)__builtin_popcountll(walked);
            wave_sync();
            if (queued >= (uint32_t)WAVE) {
                queued -= (uint32_t)WAVE;
                walk(queued, WAVE);
            }
            pc += readlane_u(incl, WAVE - 1);
            beg = readlane_u(b, WAVE - 1);
        }
        w = (int)readlane_u(incl_scan((uint32_t)w), WAVE - 1);
        if (l == 0 && w) atomicAdd(&Q.winding[k], w);
    }
    walk(0, queued);
    if ((uint32_t)l < nq) {
        const int32_t w = Q.winding[l];
        L.winding[q0 + l] = w;
        if (L.inside) L.inside[q0 + l] = L.fill_rule == 0 ? (w % 2 != 0) : (w != 0);
    }
}

// approximate_signed_area with one wave per path.  lyon's result is a serial f32 sum in
// event order, so the additions stay serial, but everything before them is spread over the
// lanes: the verbs are read 64 at a time, a lane sets one up (polynomial form, and lyon's
// serial t at every 16th point of the run, one addition per point); then the flattened
// points of a run of segments between two boundary verbs are computed 1,024 at a time, 16
// consecutive ones per lane, and each lane forms the cross products of its points with the
// points before them.  For the sum the running value goes from lane to lane, each adding its
// 16 terms.  Begin / End / Close are applied in order between the runs, with area.rs's rules
// for ill-formed paths.
//
// Bound by VALU issue, about two instructions per point, one of them the serial addition.
// 10,000 paths, 81 M points: 1,575 us when every lane set its curve up by itself (Wang's
// count, t in closed form) and terms were read lane by lane; 385 us now.
constexpr int AREA_WAVES = 4;
constexpr int AREA_RUN = 16;              // consecutive points per lane
constexpr uint32_t AREA_TABLE = 512;      // every 16th point's t: 8,192 points at once

struct AreaPoly {
    float4 a01;   // a0, a1
    float4 a23;   // a2, a3 (0 for a quadratic)
    float4 rest;  // to, step, points
};
struct AreaShared {
    AreaPoly poly[WAVE];
    uint32_t pre[WAVE + 1];  // term prefix of the window's verbs
    uint32_t pis[WAVE];      // first point of each verb
    uint32_t vbs[WAVE];      // verb codes
    float t[AREA_TABLE];     // t of the run's points 0, 16, 32, ...
};

__global__ void __launch_bounds__(WAVE* AREA_WAVES) signed_area_kernel(ValidateLaunch L) {
    __shared__ AreaShared shared[AREA_WAVES];
    const int l = lane_id();
    AreaShared& S = shared[threadIdx.x / WAVE];
    const uint32_t stride = gridDim.x * AREA_WAVES;
    for (uint32_t pid = blockIdx.x * AREA_WAVES + threadIdx.x / WAVE; pid < L.n_paths;
         pid += stride) {
        const uint32_t vb = L.verb_off[pid], nv = L.verb_off[pid + 1] - vb;
        const uint32_t pb = L.point_off[pid];
        const PathPts pts{L.points + 2ull * pb, L.point_off[pid + 1] - pb};
        float area = 0.0f, da = 0.0f;
        vec2 first = mk(0.0f, 0.0f), cur = mk(0.0f, 0.0f), v0c = mk(0.0f, 0.0f);
        bool in_sub = false, stop = false;
        uint32_t pc = 0;
        for (uint32_t c = 0; c < nv && !stop; c += WAVE) {
            const uint32_t i = c + (uint32_t)l;
            const uint32_t verb = i < nv ? (uint32_t)L.verbs[vb + i] : 0xffu;
            const uint32_t cons = points_of(verb);
            const uint32_t incl = incl_scan(cons);
            const uint32_t pi = pc + incl - cons;
            // polynomial form and flattened points (Line 1, curves Wang's count)
            uint32_t cnt = 0;
            vec2 a0 = mk(0.0f, 0.0f), a1 = a0, a2 = a0, a3 = a0, to = a0;
            float step = 1.0f;
            if (verb <= 2u) {
                const vec2 c1 = pts.at(pi);
                to = c1;
                cnt = 1;
                if (verb != 0u) {
                    a0 = pts.at(pi - 1u);
                    const vec2 c2 = pts.at(pi + 1u);
                    float n;
                    if (verb == 1u) {
                        n = quad_wang(a0, c1, c2, L.tolerance);
                        a1 = mul(sub(c1, a0), 2.0f);
                        a2 = sub(add(a0, c2), mul(c1, 2.0f));
                        to = c2;
                    } else {
                        const vec2 c3 = pts.at(pi + 2u);
                        n = cubic_wang(a0, c1, c2, c3, L.tolerance);
                        a1 = mul(sub(c1, a0), 3.0f);
                        a2 = add(sub(mul(a0, 3.0f), mul(c1, 6.0f)), mul(c2, 3.0f));
                        a3 = add(sub(c3, a0), mul(sub(c1, c2), 3.0f));
                        to = c3;
                    }
                    step = 1.0f / n;
                    cnt = seg_count(n);
                }
            }
            const uint32_t tincl = incl_scan(cnt);
            wave_sync();
            S.poly[l].a01 = make_float4(a0.x, a0.y, a1.x, a1.y);
            S.poly[l].a23 = make_float4(a2.x, a2.y, a3.x, a3.y);
            S.poly[l].rest = make_float4(to.x, to.y, step, u2f(cnt));
            S.pre[l + 1] = tincl;
            if (l == 0) S.pre[0] = 0;
            S.pis[l] = pi;
            S.vbs[l] = verb;
            wave_sync();
            const uint64_t bmask = ballot(verb >= 3u);  // boundaries and lanes past the path
            int j = 0;
            while (j < WAVE && !stop) {
                const uint32_t vj = readlane_u(verb, j);
                if (vj >= 3u) {
                    if (vj == 0xffu) break;
                    if (vj == 3u) {
                        // Begin: a sub-path starts (one inside a sub-path ends the sum)
                        if (in_sub) {
                            stop = true;
                            break;
                        }
                        first = pts.at(readlane_u(pi, j));
                        cur = first;
                        da = 0.0f;
                        v0c = mk(0.0f, 0.0f);
                        in_sub = true;
                    } else {
                        // End / Close: the closing term, then the sub-path's area
                        if (!in_sub) {
                            stop = true;
                            break;
                        }
                        da = da + cross(v0c, sub(cur, first));
                        area = area + da * 0.5f;
                        in_sub = false;
                    }
                    ++j;
                    continue;
                }
                // a run of segment verbs j .. j2 - 1, as many as the table holds (one verb
                // with more points than that takes t in closed form)
                if (!in_sub) {
                    stop = true;
                    break;
                }
                const uint64_t rest = bmask & ~mask_lt(j);
                const uint32_t r0 = readlane_u(tincl - cnt, j);
                const uint64_t over =
                    (rest | ballot(tincl - r0 > AREA_TABLE * AREA_RUN)) & ~mask_lt(j);
                int j2 = over ? __builtin_ctzll(over) : WAVE;
                const bool fits = j2 > j;
                j2 = fits ? j2 : j + 1;
                const uint32_t r1 = readlane_u(tincl, j2 - 1);
                if (fits && l >= j && l < j2) {
                    uint32_t g = tincl - cnt - r0;
                    uint32_t k = (AREA_RUN - (g & (AREA_RUN - 1))) & (AREA_RUN - 1);
                    if (k < cnt) {
                        float t = 0.0f;
                        for (uint32_t q = 0; q <= k; ++q) t = t + step;
                        for (g += k; k < cnt; k += AREA_RUN, g += AREA_RUN) {
                            S.t[g / AREA_RUN] = t;
#pragma unroll
                            for (int q = 0; q < AREA_RUN; ++q) t = t + step;
                        }
                    }
                }
                wave_sync();
                for (uint32_t q0 = r0; q0 < r1; q0 += WAVE * AREA_RUN) {
                    // lane l: points g0 .. g0 + 15 of the run (those past its end are not used)
                    const uint32_t m = r1 - q0 < (uint32_t)(WAVE * AREA_RUN)
                                           ? r1 - q0
                                           : (uint32_t)(WAVE * AREA_RUN);
                    const uint32_t g0 = q0 + (uint32_t)l * AREA_RUN;
                    float terms[AREA_RUN];
                    vec2 v1_first = mk(0.0f, 0.0f), v0 = v1_first, p = v1_first;
                    if ((uint32_t)l * AREA_RUN < m) {
                        int lo = j, hi = j2 - 1;  // last verb of the run with pre <= g0
                        while (lo < hi) {
                            const int mid = (lo + hi + 1) >> 1;
                            if (S.pre[mid] <= g0) lo = mid;
                            else hi = mid - 1;
                        }
                        int my = lo;
                        float4 a01 = S.poly[my].a01, a23 = S.poly[my].a23, re = S.poly[my].rest;
                        uint32_t end = S.pre[my + 1];
                        bool cubic = S.vbs[my] == 2u;
                        float t = fits ? S.t[(g0 - r0) / AREA_RUN]
                                       : tchain(re.z, g0 - S.pre[my] + 1u);
#pragma unroll
                        for (int u = 0; u < AREA_RUN; ++u) {
                            const uint32_t g = g0 + (uint32_t)u;
                            if (u && g >= end && my + 1 < j2) {
                                ++my;
                                a01 = S.poly[my].a01;
                                a23 = S.poly[my].a23;
                                re = S.poly[my].rest;
                                end = S.pre[my + 1];
                                cubic = S.vbs[my] == 2u;
                                t = 0.0f + re.z;
                            }
                            vec2 v = mk(a01.x, a01.y);
                            float tt = t;
                            v = add(v, mul(mk(a01.z, a01.w), tt));
                            tt = tt * t;
                            v = add(v, mul(mk(a23.x, a23.y), tt));
                            tt = tt * t;
                            const vec2 v3 = add(v, mul(mk(a23.z, a23.w), tt));
                            v = cubic ? v3 : v;
                            p = g + 1u >= end ? mk(re.x, re.y) : v;
                            t = t + re.z;
                            const vec2 v1 = sub(p, first);
                            if (u == 0) v1_first = v1;
                            else terms[u] = cross(v0, v1);
                            v0 = v1;
                        }
                    }
                    // the point before the lane's first: the previous lane's last, or the
                    // carry for lane 0
                    terms[0] = cross(mk(from_lane_before(v0.x, v0c.x), from_lane_before(v0.y, v0c.y)),
                                     v1_first);
                    // lyon's serial sum: after turn ln, lane ln holds the sum up to its end
                    const uint32_t full = m / AREA_RUN, left = m % AREA_RUN;
                    float sum = da;
                    for (uint32_t ln = 0; ln < full; ++ln) {
                        sum = from_lane_before(sum, da);
#pragma unroll
                        for (int u = 0; u < AREA_RUN; ++u) sum = sum + terms[u];
                    }
                    if (left) {
                        sum = from_lane_before(sum, da);
#pragma unroll
                        for (int u = 0; u < AREA_RUN; ++u)
                            if ((uint32_t)u < left) sum = sum + terms[u];
                    }
                    da = readlane_f(sum, (int)((m - 1) / AREA_RUN));
                    v0c = readlane_v(v0, WAVE - 1);  // of a full chunk
                }
                // a run ends at its last segment's end
                cur = readlane_v(to, j2 - 1);
                v0c = sub(cur, first);
                j = j2;
            }
            pc += readlane_u(incl, WAVE - 1);
            wave_sync();
        }
        if (l == 0) L.areas[pid] = area;
    }
}

}  // namespace lyg

extern "C" {

hipError_t lyg_launch_winding(const lyg::ValidateLaunch* L, hipStream_t s) {
    if (L->n_queries == 0) return hipSuccess;
    // queries per wave: one while 8,192 waves (8 per SIMD) can take them all, at most 64
    const uint32_t want = (L->n_queries - 1u) / 8192u + 1u;
    const uint32_t per_wave = want < (uint32_t)lyg::WAVE ? want : (uint32_t)lyg::WAVE;
    const uint32_t waves = (L->n_queries - 1u) / per_wave + 1u;
    hipLaunchKernelGGL(lyg::winding_kernel, dim3((waves - 1u) / lyg::VAL_WAVES + 1u),
                       dim3(lyg::WAVE * lyg::VAL_WAVES), 0, s, *L, per_wave);
    return hipGetLastError();
}

hipError_t lyg_launch_signed_area(const lyg::ValidateLaunch* L, hipStream_t s) {
    if (L->n_paths == 0) return hipSuccess;
    uint32_t blocks = (L->n_paths + lyg::AREA_WAVES - 1) / lyg::AREA_WAVES;
    if (blocks > 65536u) blocks = 65536u;
    hipLaunchKernelGGL(lyg::signed_area_kernel, dim3(blocks), dim3(lyg::WAVE * lyg::AREA_WAVES), 0,
                       s, *L);
    return hipGetLastError();
}


}  // extern "C"
