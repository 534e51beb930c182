// Decoding of one path verb into its flattened points: the counts, the polynomial forms and
// the exact last points (shared by the fixed-width and the variable-width stroke kernels).
#pragma once
#include "lyg_math.h"
#include "stroke_core.h"

namespace lyg {

enum : uint32_t {
    K_BEGIN = 1u,
    K_LINE = 2u,
    K_QUAD = 3u,
    K_CUBIC = 4u,
    K_END = 5u,
};

struct VRec {
    vec2 a0, a1, a2, a3;  // curve A polynomial form (quadratic: a3 unused)
    vec2 b0, b1, b2;      // curve B (second half of a split quadratic)
    vec2 toA, toB;        // exact last points; BEGIN/LINE keep their point in toA
    float sA, sB;         // flattening step 1/n
    uint32_t nA, nB;      // flattened point counts
    uint32_t off;         // first step of this verb in the chunk
    uint32_t kind;        // K_* | (close << 8)
};

__device__ __forceinline__ vec2 ldp(const float* pts, uint32_t n, uint32_t i) {
    if (i >= n) return mk(__builtin_nanf(""), __builtin_nanf(""));
    const float2 v = reinterpret_cast<const float2*>(pts)[i];
    return mk(v.x, v.y);
}

__device__ __forceinline__ vec2 horner(const VRec& r, bool b, bool cubic, float t) {
    vec2 v = b ? r.b0 : r.a0;
    float tt = t;
    v = add(v, mul(b ? r.b1 : r.a1, tt));
    tt = tt * t;
    v = add(v, mul(b ? r.b2 : r.a2, tt));
    if (cubic) {
        tt = tt * t;
        v = add(v, mul(r.a3, tt));
    }
    return v;
}

// Decode verb `vi` of the path into rec.  `p` is the index of its first point.  `split`:
// where a quadratic's split parameter goes (not positive when it is not split).
__device__ __forceinline__ void decode_verb(uint8_t verb, const float* pts, uint32_t npts,
                                            uint32_t p, float tol, VRec& r,
                                            float* split = nullptr) {
    const float nan = __builtin_nanf("");
    r.nA = 0;
    r.nB = 0;
    r.sA = r.sB = 0.0f;
    r.a0 = r.a1 = r.a2 = r.a3 = mk(0.0f, 0.0f);
    r.b0 = r.b1 = r.b2 = mk(0.0f, 0.0f);
    r.toA = r.toB = mk(nan, nan);
    vec2 from = p > 0 ? ldp(pts, npts, p - 1) : mk(nan, nan);
    switch (verb) {
        case LYG_VERB_BEGIN:
            r.kind = K_BEGIN;
            r.toA = ldp(pts, npts, p);
            r.nA = 1;
            break;
        case LYG_VERB_LINE:
            r.kind = K_LINE;
            r.toA = ldp(pts, npts, p);
            r.nA = 1;
            break;
        case LYG_VERB_QUADRATIC: {
            r.kind = K_QUAD;
            vec2 ctrl = ldp(pts, npts, p), to = ldp(pts, npts, p + 1);
            float ts = find_sharp_turn(from, ctrl, to);
            if (split) *split = ts;
            vec2 A0 = from, A1 = ctrl, A2 = to;
            if (ts > 0.0f) {
                // QuadraticBezierSegment::split (quadratic_bezier.rs:208-223)
                vec2 sp = quad_sample(from, ctrl, to, ts);
                A1 = lerp(from, ctrl, ts);
                A2 = sp;
                vec2 B0 = sp, B1 = lerp(ctrl, to, ts), B2 = to;
                float nb = quad_wang(B0, B1, B2, tol);
                r.sB = 1.0f / nb;
                r.nB = seg_count(nb);
                r.b0 = B0;
                r.b1 = mul(sub(B1, B0), 2.0f);
                r.b2 = sub(add(B0, B2), mul(B1, 2.0f));
                r.toB = B2;
            }
            float na = quad_wang(A0, A1, A2, tol);
            r.sA = 1.0f / na;
            r.nA = seg_count(na);
            r.a0 = A0;
            r.a1 = mul(sub(A1, A0), 2.0f);
            r.a2 = sub(add(A0, A2), mul(A1, 2.0f));
            r.toA = A2;
            break;
        }
        case LYG_VERB_CUBIC: {
            r.kind = K_CUBIC;
            vec2 c1 = ldp(pts, npts, p), c2 = ldp(pts, npts, p + 1), to = ldp(pts, npts, p + 2);
            float n = cubic_wang(from, c1, c2, to, tol);
            r.sA = 1.0f / n;
            r.nA = seg_count(n);
            // polynomial_form (cubic_bezier.rs:1318-1325)
            r.a0 = from;
            r.a1 = mul(sub(c1, from), 3.0f);
            r.a2 = add(sub(mul(from, 3.0f), mul(c1, 6.0f)), mul(c2, 3.0f));
            r.a3 = add(sub(to, from), mul(sub(c1, c2), 3.0f));
            r.toA = to;
            break;
        }
        case LYG_VERB_CLOSE:
            r.kind = K_END | (1u << 8);
            r.nA = 1;
            break;
        default:  // END
            r.kind = K_END;
            r.nA = 1;
            break;
    }
}

// lyon's serial t (t = t + step from 0) of a chunk's curve steps [b0, b0 + T_SPAN) at every
// 16th step of the chunk: a lane per verb adds its curve's steps up, one addition per step (the
// closed form once, where a curve starts far before b0), and a window's lanes then need 15
// additions at most.  b0 is a multiple of 16; steps from b1 on are left out.
static constexpr uint32_t T_SPAN = 4096;
__device__ __forceinline__ void t_table(float* tab, const VRec& r, bool in, uint32_t b0,
                                        uint32_t b1) {
    const uint32_t kind = r.kind & 0xffu;
    if (!in || (kind != K_QUAD && kind != K_CUBIC)) return;
    if (b1 - b0 > T_SPAN) b1 = b0 + T_SPAN;
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
        const uint32_t start = half ? r.off + r.nA : r.off, n = half ? r.nB : r.nA;
        const float step = half ? r.sB : r.sA;
        const uint32_t lo = ((start > b0 ? start : b0) + 15u) & ~15u;
        const uint32_t hi = start + n < b1 ? start + n : b1;
        if (lo >= hi) continue;
        const uint32_t j = lo - start + 1u;
        float t = 0.0f;
        if (j <= 64u) {
            for (uint32_t q = 0; q < j; ++q) t = t + step;
        } else {
            t = tchain(step, j);
        }
        for (uint32_t g = lo; g < hi; g += 16u) {
            tab[(g - b0) >> 4] = t;
#pragma unroll
            for (int q = 0; q < 16; ++q) t = t + step;
        }
    }
}
// t of the chunk's step g, the j-th (from 1) of its curve, from a table of b0 on.
__device__ __forceinline__ float t_at(const float* tab, uint32_t b0, uint32_t g, uint32_t j,
                                      float step) {
    const uint32_t ahead = g & 15u;
    const bool listed = j > ahead;  // the curve holds the listed step before g
    float t = listed ? tab[((g - b0) >> 4) & (T_SPAN / 16u - 1u)] : 0.0f;
    const uint32_t more = listed ? ahead : j;
#pragma unroll
    for (uint32_t q = 0; q < 15u; ++q) t = q < more ? t + step : t;
    return t;
}

__device__ __forceinline__ uint32_t verb_points(uint8_t v) {
    switch (v) {
        case LYG_VERB_BEGIN:
        case LYG_VERB_LINE:
        case LYG_VERB_CLOSE:
            return 1;
        case LYG_VERB_QUADRATIC:
            return 2;
        case LYG_VERB_CUBIC:
            return 3;
        default:
            return 0;
    }
}

}  // namespace lyg
