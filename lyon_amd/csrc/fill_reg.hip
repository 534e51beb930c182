// Fill sweep for gfx950 with the sweep's state in registers, and the triangulation of its
// spans as work of its own.
//
// The sweep (fill.rs:836-867) is one serial chain per path, so what bounds it is the latency
// of an event.  One wave sweeps one path, as the kernel over arrays in memory does
// (fill.hip, which still takes the paths that outgrow this one), with these differences:
//   * active edge i is held by lane i mod 64 in register set i / 64: locating the point,
//     checking the rest and searching intersections read nothing from memory, an event that
//     replaces as many edges as it removes moves nothing, and others shift lanes;
//   * edges below the event, the sorted events ahead (64 at a time) and the pending pushes
//     and span operations of the event are lanes of registers too, read back as scalars;
//   * pending intersections: 64 columns in LDS, one per lane, each lane keeping the earliest
//     of its column; the next event is a wave minimum over the lanes, and taking one looks
//     at one column only;
//   * the monotone triangulation is left out of the chain: the sweep writes a log of span
//     operations (begin, vertex on a side, end), linked per span, and lanes walk the spans
//     afterwards, all at once; after a scan of the operations' triangles in log order, they
//     go where the sweep would have written them.
// Vertices, triangles and their order are those of the sweep over arrays.
//
// A path stops with a retry status when it has more than 64 C active edges (or spans) or more
// pending intersections than its columns hold, which a launch of more may, or more than 64 edges
// below one event (spans it ends, pushes), which is left to the sweep over arrays.
#include <hip/hip_runtime.h>

#include "fill_core.h"
#include "lyg_math.h"
#include "lyg_types.h"
#include "wave.h"

namespace lyg {

namespace fillk {

enum : uint32_t { OP_LEFT = 0u, OP_RIGHT = 1u, OP_BEGIN = 2u, OP_END = 3u };
static constexpr uint32_t DEAD = 0xffffffffu;  // a span that ended, until the next cleanup
static constexpr uint32_t MERGE_BIT = 0x10000u;

// A value that is the same in every lane, as a scalar.  The sweep's control flow is uniform, but
// the compiler takes a value for divergent when it is loaded from LDS through a lane, or when
// its definition meets a lane's branch (lane 0 stores, others do not) in one block; every
// branch that depends on it then works on lane masks with the state in vector registers
// (measured: 22,000-28,000 cycles per event, against 7,600-21,200 with the scalars kept scalar).  So
// lanes take values by selects, not branches, and counters pass through here where they change.
__device__ __forceinline__ uint32_t uni(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}
__device__ __forceinline__ float unif(float v) { return u2f(uni(f2u(v))); }
__device__ __forceinline__ bool unib(bool v) { return uni(v ? 1u : 0u) != 0u; }
__device__ __forceinline__ int32_t wind_of(uint32_t wm) { return (int32_t)(int16_t)(wm & 0xffffu); }

// Element p of values held 64 per register.
template <int C>
__device__ __forceinline__ uint32_t rget(const uint32_t (&r)[C], uint32_t p) {
    uint32_t v = r[0];
    if (C > 1 && p >= (uint32_t)WAVE) {
#pragma unroll
        for (int c = 1; c < C; ++c) v = (p >> 6) == (uint32_t)c ? r[c] : v;
    }
    return readlane_u(v, (int)(p & 63u));
}
template <int C>
__device__ __forceinline__ float rgetf(const float (&r)[C], uint32_t p) {
    float v = r[0];
    if (C > 1 && p >= (uint32_t)WAVE) {
#pragma unroll
        for (int c = 1; c < C; ++c) v = (p >> 6) == (uint32_t)c ? r[c] : v;
    }
    return readlane_f(v, (int)(p & 63u));
}
template <int C, class T>
__device__ __forceinline__ void rset(T (&r)[C], uint32_t p, T x) {
    const uint32_t l = (uint32_t)lane_id();
#pragma unroll
    for (int c = 0; c < C; ++c) r[c] = (uint32_t)c * 64u + l == p ? x : r[c];
}
__device__ __forceinline__ uint32_t perm(uint32_t v, int src4) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute(src4, (int)v);
}
__device__ __forceinline__ float perm(float v, int src4) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_ds_bpermute(src4, __builtin_bit_cast(int, v)));
}
// Elements [from, n) move up by d (1-63) places; n: elements after the move.
template <int C, class T>
__device__ __forceinline__ void rshift_up(T (&r)[C], uint32_t from, uint32_t n, uint32_t d) {
    const uint32_t l = (uint32_t)lane_id();
    const int src = (int)(((l - d) & 63u) << 2);
    T below = r[0];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        if ((uint32_t)c * 64u >= n) break;
        const T q = perm(r[c], src);
        const T x = l >= d ? q : below;
        below = q;
        r[c] = (uint32_t)c * 64u + l >= from + d ? x : r[c];
    }
}
// Elements [from + d, n) move down by d (1-63) places.
template <int C, class T>
__device__ __forceinline__ void rshift_down(T (&r)[C], uint32_t from, uint32_t n, uint32_t d) {
    const uint32_t l = (uint32_t)lane_id();
    const int src = (int)(((l + d) & 63u) << 2);
    T cur = perm(r[0], src);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        if ((uint32_t)c * 64u >= n) break;
        T nxt = cur;
        if (c + 1 < C) nxt = perm(r[c + 1 < C ? c + 1 : c], src);
        const T x = l + d < 64u ? cur : nxt;
        cur = nxt;
        r[c] = (uint32_t)c * 64u + l >= from ? x : r[c];
    }
}

// The columns of pending events in LDS: entry e of lane l's column at [64 e + l].
struct Cols {
    float2* pos;
    float2* to;
    uint2* meta;   // insertion sequence, winding (low 16 bits) | edge << 16
    uint32_t rows;
};
__host__ __device__ inline size_t cols_bytes(uint32_t rows) { return 24ull * 64ull * rows; }

template <int C>
__device__ __forceinline__ void reg_sweep(const FillLaunch& L, uint32_t path, uint32_t k,
                                          uint8_t* work, const Cols& H, uint32_t* hist,
                                          uint32_t* out_status, uint32_t* out_nv,
                                          uint32_t* out_ops, uint32_t* out_hint) {
    const int lane = lane_id();
    const uint32_t ul = (uint32_t)lane;
    const lyg_fill_options o = L.opts[L.opts_stride ? path : 0];
    const uint32_t rule = uni(o.fill_rule);
    const bool horiz = uni(o.sweep_orientation) == LYG_ORIENT_HORIZONTAL;
    const bool crossings = uni(o.handle_intersections) != 0u;
    const float tolerance = unif(o.tolerance);
    const float tol = tolerance * 0.5f;  // fill.rs:772-778
    *out_nv = *out_ops = 0;
    if (!(tolerance > 0.0f)) {  // tessellate_impl (fill.rs:755-759)
        *out_status = ST_TOLERANCE_NAN;
        return;
    }
    Sweep g;  // the event builder's view
    g.lane = lane;
    g.lds_only = true;
    g.status = ST_OK;
    carve(work, nullptr, 0, L.caps, g.w);
    const uint32_t made = uni(make_events(g, L.in, path, o, hist));
    if (made != ST_OK) {
        *out_status = made;
        return;
    }
    const uint32_t n_static = uni(g.n_static);
    const uint64_t* skey = g.w.key_a;
    const uint32_t* sidx = g.w.idx_a;
    const Ev* sev = g.w.ev;
    const uint32_t act_cap = min(64u * (uint32_t)C, L.act_limit);
    const uint32_t heap_cap = min(64u * H.rows, L.heap_limit);
    float2* out_v = reinterpret_cast<float2*>(L.stage_v) + L.stage_v_off[k];
    const uint32_t vcap = uni((uint32_t)(L.stage_v_off[k + 1] - L.stage_v_off[k]));
    FillOp* ops = L.ops + L.stage_t_off[k];
    const uint32_t op_cap = uni((uint32_t)(L.stage_t_off[k + 1] - L.stage_t_off[k]));

    // the status of a path that outgrows the sets, or the columns
    const uint32_t MORE_SETS = C < (int)REG_MAX_SETS ? ST_RETRY_SETS : ST_RETRY_ARRAYS;
    const uint32_t MORE_ROWS = H.rows < REG_MAX_ROWS ? ST_RETRY_SETS : ST_RETRY_ARRAYS;
    uint32_t status = ST_OK;
    auto fail = [&](uint32_t st) { status = uni(status == ST_OK ? st : status); };
    // active edges (fill.rs:153-170): winding (low 16 bits) | merge, first vertex id
    float fx[C], fy[C], tx[C], ty[C];
    uint32_t wm[C], fid[C], span[C];  // span: its last operation, or DEAD
#pragma unroll
    for (int c = 0; c < C; ++c) {
        fx[c] = fy[c] = tx[c] = ty[c] = 0.0f;
        wm[c] = fid[c] = span[c] = 0;
    }
    uint32_t n_act = 0, n_spans = 0, n_ops = 0, nv = 0;
    // pending events: this lane's column and its earliest entry
    uint32_t h_cnt = 0, h_hi = ~0u, h_lo = ~0u, h_seq = ~0u, h_row = 0;
    float h_px = 0.0f, h_py = 0.0f;
    uint32_t heap_n = 0, heap_seq = 0, level = 0;  // level: no column is shorter
    // sorted events [s_base, s_base + 64)
    uint32_t cur = 0, s_base = 0;
    float s_px = 0.0f, s_py = 0.0f, s_tx = 0.0f, s_ty = 0.0f;
    uint32_t s_hi = 0, s_lo = 0, s_w = 0;
    auto load_static = [&](uint32_t base) {
        const uint32_t j = base + ul;
        if (j < n_static) {
            const uint64_t key = skey[j];
            const Ev e = ld(&sev[sidx[j]]);
            s_hi = (uint32_t)(key >> 32);
            s_lo = (uint32_t)key;
            s_px = e.pos.x;
            s_py = e.pos.y;
            s_tx = e.to.x;
            s_ty = e.to.y;
            s_w = ((uint32_t)e.winding & 0xffffu) | (e.is_edge << 16);
        }
        s_base = uni(base);
    };
    load_static(0);
    // edges below the event (fill.rs:302-310), one per lane
    float b_tx = 0.0f, b_ty = 0.0f, b_key = 0.0f;
    uint32_t b_w = 0, n_below = 0;
    // pushes and span operations of the event, one per lane
    float q_px = 0.0f, q_py = 0.0f, q_tx = 0.0f, q_ty = 0.0f;
    uint32_t q_w = 0, n_push = 0;
    float a_x = 0.0f, a_y = 0.0f;
    uint32_t a_id = 0, a_op = 0, n_acts = 0;  // a_op: kind | span index << 2
    int32_t a_span = 0;
    vec2 cp = mk(0.0f, 0.0f);
    uint32_t cv = 0;
    auto add_below = [&](vec2 to, int32_t w) {
        if (n_below >= (uint32_t)WAVE) {
            fail(ST_RETRY_ARRAYS);
            return;
        }
        const float key = slope(sub(to, cp));
        const bool me = ul == n_below;
        b_tx = me ? to.x : b_tx;
        b_ty = me ? to.y : b_ty;
        b_key = me ? key : b_key;
        b_w = me ? (uint32_t)w : b_w;
        n_below = uni(n_below + 1u);
    };
    auto push_later = [&](vec2 pos, vec2 to, int32_t w, bool edge) {
        if (n_push >= (uint32_t)WAVE) {
            fail(ST_RETRY_ARRAYS);
            return;
        }
        const bool me = ul == n_push;
        q_px = me ? pos.x : q_px;
        q_py = me ? pos.y : q_py;
        q_tx = me ? to.x : q_tx;
        q_ty = me ? to.y : q_ty;
        q_w = me ? ((uint32_t)w & 0xffffu) | (edge ? MERGE_BIT : 0u) : q_w;
        n_push = uni(n_push + 1u);
    };
    auto span_op = [&](uint32_t kind, int32_t idx, vec2 pos, uint32_t id) {
        if (n_acts >= (uint32_t)WAVE) {
            fail(ST_RETRY_ARRAYS);
            return;
        }
        const bool me = ul == n_acts;
        a_x = me ? pos.x : a_x;
        a_y = me ? pos.y : a_y;
        a_id = me ? id : a_id;
        a_op = me ? kind : a_op;
        a_span = me ? idx : a_span;
        n_acts = uni(n_acts + 1u);
    };
    // Spans::begin_span / the tessellators' vertex and end (fill.rs:200-300): the queued span
    // operations go to the log.  A single ended span keeps its slot until the next begin
    // takes it (an event at a crossing ends and begins the span between the same two) or the
    // queue is through.
    auto run_span_ops = [&]() {
        uint32_t n_dead = 0, dead_at = 0;
        auto drop_dead = [&]() {
            if (n_dead == 1u) {
                rshift_down(span, dead_at, n_spans, 1u);
                n_spans -= 1u;
            } else {
                for (uint32_t i = n_spans; i-- > 0u;)
                    if (rget(span, i) == DEAD) {
                        rshift_down(span, i, n_spans, 1u);
                        n_spans -= 1u;
                    }
            }
            n_dead = 0;
        };
        bool closing = true;  // still in the vertices and ends above the event
        for (uint32_t q = 0; q < n_acts && status == ST_OK; ++q) {
            const uint32_t kind = readlane_u(a_op, (int)q);
            const int32_t idx = (int32_t)readlane_u((uint32_t)a_span, (int)q);
            const vec2 pos = readlane_v(mk(a_x, a_y), (int)q);
            const uint32_t id = readlane_u(a_id, (int)q);
            uint32_t link = DEAD;
            const bool reuse = kind == OP_BEGIN && n_dead == 1u && (uint32_t)idx == dead_at;
            if (kind == OP_BEGIN) {
                if (!reuse) {
                    if (n_dead) drop_dead();
                    if (idx < 0 || (uint32_t)idx > n_spans) {
                        fail(ST_INTERNAL);
                        break;
                    }
                    if (n_spans + 1u > 64u * (uint32_t)C) {
                        fail(MORE_SETS);
                        break;
                    }
                }
                closing = false;
            } else {
                // a vertex after the ends (a split event's) sees the spans cleaned up
                if (!closing && n_dead) drop_dead();
                if (idx < 0 || (uint32_t)idx >= n_spans) {
                    fail(ST_INTERNAL);
                    break;
                }
                link = rget(span, (uint32_t)idx);
                if (link == DEAD) {
                    fail(ST_INTERNAL);
                    break;
                }
            }
            const uint32_t op = n_ops++;
            if (op >= op_cap) {
                fail(ST_RETRY);
                break;
            }
            if (lane == 0) {
                float4* d = reinterpret_cast<float4*>(ops + op);
                d[0] = make_float4(pos.x, pos.y, u2f(id), u2f(kind));
                d[1] = make_float4(u2f(DEAD), u2f(DEAD), u2f(DEAD), 0.0f);
            }
            if (lane == 0 && link != DEAD) ops[link].next = op;
            if (kind == OP_BEGIN) {
                if (reuse) {
                    n_dead = 0;
                } else {
                    rshift_up(span, (uint32_t)idx, n_spans + 1u, 1u);
                    n_spans += 1u;
                }
                rset(span, (uint32_t)idx, op);
            } else if (kind == OP_END) {
                rset(span, (uint32_t)idx, DEAD);
                dead_at = (uint32_t)idx;
                ++n_dead;
            } else {
                rset(span, (uint32_t)idx, op);
            }
            n_dead = uni(n_dead);
            dead_at = uni(dead_at);
            n_spans = uni(n_spans);
            n_ops = uni(n_ops);
        }
        if (n_dead) drop_dead();
        n_spans = uni(n_spans);
        n_acts = 0;
    };

    for (;;) {
        status = uni(status);
        cur = uni(cur);
        s_base = uni(s_base);
        heap_n = uni(heap_n);
        heap_seq = uni(heap_seq);
        level = uni(level);
        nv = uni(nv);
        n_ops = uni(n_ops);
        n_act = uni(n_act);
        n_spans = uni(n_spans);
        n_below = n_push = n_acts = 0;
        if (status != ST_OK) break;
        // ---- the next position (tessellator_loop, fill.rs:836-867) ----
        if (cur - s_base >= 64u && cur < n_static) load_static(cur);
        const bool hs = cur < n_static;
        if (!hs && heap_n == 0u) break;
        uint32_t k_hi = ~0u, k_lo = ~0u;
        if (hs) {
            k_hi = readlane_u(s_hi, (int)(cur - s_base));
            k_lo = readlane_u(s_lo, (int)(cur - s_base));
            cp = readlane_v(mk(s_px, s_py), (int)(cur - s_base));
        }
        if (heap_n) {
            const uint32_t t_hi = wave_min_u32(h_hi);
            uint64_t m = ballot(h_hi == t_hi && h_cnt != 0u);
            uint32_t t_lo;
            if (__builtin_popcountll(m) == 1) {
                t_lo = readlane_u(h_lo, __builtin_ctzll(m));
            } else {
                t_lo = wave_min_u32(h_hi == t_hi && h_cnt != 0u ? h_lo : ~0u);
                m = ballot(h_hi == t_hi && h_lo == t_lo && h_cnt != 0u);
            }
            if (!hs || t_hi < k_hi || (t_hi == k_hi && t_lo < k_lo)) {
                k_hi = t_hi;
                k_lo = t_lo;
                // the earliest inserted of the entries at this key gives the position
                int t = __builtin_ctzll(m);
                if (__builtin_popcountll(m) > 1) {
                    const uint32_t sq = wave_min_u32((m >> lane) & 1ull ? h_seq : ~0u);
                    t = __builtin_ctzll(ballot(((m >> lane) & 1ull) && h_seq == sq));
                }
                cp = readlane_v(mk(h_px, h_py), t);
            }
        }
        cv = nv;
        nv += 1u;
        if (cv >= vcap) {
            fail(ST_RETRY);
            break;
        }
        // fill.rs:890-894
        if (lane == 0) out_v[cv] = horiz ? make_float2(cp.y, -cp.x) : make_float2(cp.x, cp.y);
        // ---- initialize_events: the edges below from every event at this position ----
        while (cur < n_static && status == ST_OK) {
            if (cur - s_base >= 64u) load_static(cur);
            const int e = (int)(cur - s_base);
            if (readlane_u(s_hi, e) != k_hi || readlane_u(s_lo, e) != k_lo) break;
            const uint32_t w = readlane_u(s_w, e);
            if (w & MERGE_BIT) add_below(readlane_v(mk(s_tx, s_ty), e), wind_of(w));
            ++cur;
        }
        while (heap_n && status == ST_OK) {
            const uint64_t m = ballot(h_cnt != 0u && h_hi == k_hi && h_lo == k_lo);
            if (!m) break;
            int t = __builtin_ctzll(m);
            if (__builtin_popcountll(m) > 1) {
                const uint32_t sq = wave_min_u32((m >> lane) & 1ull ? h_seq : ~0u);
                t = __builtin_ctzll(ballot(((m >> lane) & 1ull) && h_seq == sq));
            }
            // take column t's earliest entry: its last entry fills the gap, and the rest of
            // the column is looked through by the wave, one entry per lane
            const uint32_t row = readlane_u(h_row, t), last = readlane_u(h_cnt, t) - 1u;
            const float2 l_to = H.to[64u * row + (uint32_t)t];
            const vec2 eto = mk(unif(l_to.x), unif(l_to.y));
            const uint32_t ew = uni(H.meta[64u * row + (uint32_t)t].y);
            float2 cpos = make_float2(0.0f, 0.0f), cto = cpos;
            uint2 cm = make_uint2(~0u, 0u);
            const bool in = ul <= last && ul != row;
            if (in) {
                cpos = H.pos[64u * ul + (uint32_t)t];
                cto = H.to[64u * ul + (uint32_t)t];
                cm = H.meta[64u * ul + (uint32_t)t];
            }
            wave_sync();
            if (in && ul == last) {
                H.pos[64u * row + (uint32_t)t] = cpos;
                H.to[64u * row + (uint32_t)t] = cto;
                H.meta[64u * row + (uint32_t)t] = cm;
            }
            wave_sync();
            uint32_t m_hi = ~0u, m_lo = ~0u, m_seq = ~0u, m_row = 0;
            float m_px = 0.0f, m_py = 0.0f;
            if (last > 0u) {
                const uint32_t c_hi = fkey(cpos.y), c_lo = fkey(cpos.x);
                m_hi = wave_min_u32(in ? c_hi : ~0u);
                uint64_t mm = ballot(in && c_hi == m_hi);
                if (__builtin_popcountll(mm) > 1) {
                    const uint32_t lo = wave_min_u32(in && c_hi == m_hi ? c_lo : ~0u);
                    mm = ballot(in && c_hi == m_hi && c_lo == lo);
                    if (__builtin_popcountll(mm) > 1) {
                        const uint32_t sq = wave_min_u32((mm >> lane) & 1ull ? cm.x : ~0u);
                        mm = ballot(((mm >> lane) & 1ull) && cm.x == sq);
                    }
                }
                const int sl = __builtin_ctzll(mm);
                m_lo = readlane_u(c_lo, sl);
                m_seq = readlane_u(cm.x, sl);
                m_px = readlane_f(cpos.x, sl);
                m_py = readlane_f(cpos.y, sl);
                m_row = (uint32_t)sl == last ? row : (uint32_t)sl;
            }
            const bool me = lane == t;
            h_cnt = me ? last : h_cnt;
            h_hi = me ? m_hi : h_hi;
            h_lo = me ? m_lo : h_lo;
            h_seq = me ? m_seq : h_seq;
            h_row = me ? m_row : h_row;
            h_px = me ? m_px : h_px;
            h_py = me ? m_py : h_py;
            heap_n = uni(heap_n - 1u);
            level = uni(min(level, last));
            if (ew & MERGE_BIT) add_below(eto, wind_of(ew));
        }
        n_below = uni(n_below);
        status = uni(status);
        if (status != ST_OK) break;

        // ---- process_events; on an order error recover and try once more (fill.rs:855-863)
        uint32_t above_start = 0, above_end = 0, n_split = 0;
        uint32_t sp_edge = 0;  // scan.edges_to_split, one per lane
        bool split_event = false, merge_event = false;
        WState wbp = wnew();
        for (int attempt = 0;; ++attempt) {
            // scan_active_edges (fill.rs:1045-1291)
            bool ok = true;
            n_split = 0;
            n_acts = 0;  // scan.vertex_events and spans_to_end become span operations
            merge_event = split_event = false;
            bool merge_split_event = false, connecting = false, previous_was_merge = false;
            uint32_t idx = 0;
            WState winding = wnew();
            // One pass over the edges: classify_before up to the first edge that is not
            // before the point, and for all of them whether check_remaining_edges would
            // refuse one after the point's edges.
            bool stopped = false;
            uint64_t badm[C];
#pragma unroll
            for (int c = 0; c < C; ++c) badm[c] = 0ull;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                if ((uint32_t)c * 64u >= n_act) break;
                const uint32_t nin = min(64u, n_act - (uint32_t)c * 64u);
                const uint64_t plainm = ballot((ul < nin) & ((wm[c] & MERGE_BIT) == 0u));
                const float mn = ffmin(fx[c], tx[c]), mx = fmax_(fx[c], tx[c]);
                const uint64_t at_to = ballot((cp.x == tx[c]) & (cp.y == ty[c])) & plainm;
                const uint64_t left = ballot(mx < cp.x) & plainm;
                const uint64_t span_x = plainm & ~at_to & ~left & ~ballot(mn > cp.x);
                uint64_t beforem = left & ~at_to, connm = at_to;
                badm[c] = at_to | left;
                float x = 0.0f;
                if (span_x) {
                    const float dy = ty[c] - fy[c];
                    const float q = (cp.y - fy[c]) / dy, t = dy == 0.0f ? 0.0f : q;
                    x = ffmin(ffmax(fx[c] * (1.0f - t) + tx[c] * t, mn), mx);
                    const uint64_t hit =
                        ballot((fy[c] == ty[c]) | (ffabs(x - cp.x) <= tol)) & span_x;
                    connm |= hit;
                    beforem |= span_x & ~hit & ~ballot(x > cp.x);
                    badm[c] |= span_x & ballot((mn < cp.x) & (x < cp.x));
                }
                if (stopped) continue;
                const uint64_t stopm = plainm & ~beforem;
                const uint32_t nproc = stopm ? (uint32_t)__builtin_ctzll(stopm) : nin;
                // the winding after each edge before the point: +1 and -1 edges by counting
                // the masks below a lane, others by a scan
                const int32_t wl = wind_of(wm[c]);
                const uint64_t take = plainm & mask_lt((int)nproc);
                const uint64_t pos = ballot(wl == 1) & take, neg = ballot(wl == -1) & take;
                int32_t number;
                if (!(take & ~(pos | neg | ballot(wl == 0)))) {
                    const uint32_t np = __builtin_amdgcn_mbcnt_hi(
                        (uint32_t)(pos >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)pos, 0u));
                    const uint32_t nn = __builtin_amdgcn_mbcnt_hi(
                        (uint32_t)(neg >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)neg, 0u));
                    number = winding.number + (int32_t)np - (int32_t)nn + wl;
                    winding.number = (int16_t)(winding.number + __builtin_popcountll(pos) -
                                               __builtin_popcountll(neg));
                } else {
                    const uint32_t incl = incl_scan((take >> lane) & 1ull ? (uint32_t)wl : 0u);
                    number = winding.number + (int32_t)incl;
                    winding.number =
                        (int16_t)(winding.number + (int32_t)readlane_u(incl, WAVE - 1));
                }
                const uint64_t mergem = ~plainm & mask_lt((int)nproc);
                winding.span_index +=
                    (int32_t)__builtin_popcountll(ballot(rule_in(rule, number)) & take) +
                    (int32_t)__builtin_popcountll(mergem);
                if (nproc > 0u) {
                    winding.in = rule_in(rule, winding.number);
                    previous_was_merge = ((mergem >> (nproc - 1u)) & 1ull) != 0;
                }
                idx = (uint32_t)c * 64u + nproc;
                if (stopm) {
                    stopped = true;
                    connecting = ((connm >> nproc) & 1ull) != 0;
                }
            }
            idx = uni(idx);
            winding.number = (int32_t)uni((uint32_t)winding.number);
            winding.span_index = (int32_t)uni((uint32_t)winding.span_index);
            above_start = idx;
            wbp = winding;
            if (previous_was_merge) {
                wbp.span_index -= 1;
                above_start -= 1;
                if (!connecting) {
                    span_op(OP_RIGHT, winding.span_index - 1, cp, cv);
                    span_op(OP_LEFT, winding.span_index, cp, cv);
                    merge_split_event = true;
                }
            }
            split_event = !connecting && winding.in && !merge_split_event;
            uint32_t n_end = 0;
            int32_t end_span_of = 0;  // scan.spans_to_end, one per lane
            if (connecting) {
                const bool in_before = winding.in;
                bool first = !previous_was_merge, more = true;
                while (more && ok && idx < n_act) {
                    // is_edge_connecting of 64 edges at once, then their run in order
                    const uint32_t cc = idx >> 6;
                    float ex0 = fx[0], ey0 = fy[0], ex1 = tx[0], ey1 = ty[0];
                    uint32_t ewm = wm[0];
#pragma unroll
                    for (int c = 1; c < C; ++c)
                        if (cc == (uint32_t)c) {
                            ex0 = fx[c];
                            ey0 = fy[c];
                            ex1 = tx[c];
                            ey1 = ty[c];
                            ewm = wm[c];
                        }
                    const bool at_to = (cp.x == ex1) & (cp.y == ey1);
                    const float mn = ffmin(ex0, ex1), mx = fmax_(ex0, ex1);
                    const bool gone = (mx + tol < cp.x) | (ey1 < cp.y);
                    const float dy = ey1 - ey0;
                    const float q = (cp.y - ey0) / dy, t = dy == 0.0f ? 0.0f : q;
                    const float x = ffmin(ffmax(ex0 * (1.0f - t) + ex1 * t, mn), mx);
                    const float flat = ((mx >= cp.x) & (mn <= cp.x)) ? cp.x : ex1;
                    const float ex = ey0 != ey1 ? x : flat;
                    const bool past = mn > cp.x;
                    const bool near = ffabs(ex - cp.x) <= tol;
                    const uint64_t mm = ballot((ewm & MERGE_BIT) != 0u);
                    const uint64_t splitm = ballot(!at_to & !gone & !past & near);
                    const uint64_t connm = ballot(at_to) | splitm;
                    const uint64_t badm =
                        ballot(!at_to & (gone | (!past & !near & (ex < cp.x))));
                    for (int b = (int)(idx & 63u); b < WAVE && idx < n_act; ++b) {
                        if ((mm >> b) & 1ull) {
                            if (!winding.in) {  // MergeVertexOutside
                                ok = false;
                                break;
                            }
                            end_span_of = ul == n_end ? winding.span_index : end_span_of;
                            ++n_end;
                            winding.span_index += 1;
                            idx += 1u;
                            first = false;
                            continue;
                        }
                        if ((badm >> b) & 1ull) {
                            ok = false;
                            break;
                        }
                        if (!((connm >> b) & 1ull)) {
                            more = false;
                            break;
                        }
                        if ((splitm >> b) & 1ull) {
                            sp_edge = ul == n_split ? idx : sp_edge;
                            ++n_split;
                        }
                        if (!first && winding.in) {
                            end_span_of = ul == n_end ? winding.span_index : end_span_of;
                            ++n_end;
                        }
                        wupdate(winding, rule, wind_of(readlane_u(ewm, b)));
                        if (winding.in && winding.span_index >= (int32_t)n_spans) {
                            ok = false;
                            break;
                        }
                        idx += 1u;
                        first = false;
                    }
                    if (n_end > (uint32_t)WAVE || n_split > (uint32_t)WAVE) {
                        fail(ST_RETRY_ARRAYS);
                        break;
                    }
                }
                if (status != ST_OK) break;
                if (ok) {
                    const bool in_after = winding.in;
                    if (in_before && in_after && n_below == 0u && n_split == 0u) merge_event = true;
                    if (in_before) span_op(OP_RIGHT, wbp.span_index, cp, cv);
                    if (in_after) span_op(OP_LEFT, winding.span_index, cp, cv);
                    for (uint32_t e = 0; e < n_end; ++e)
                        span_op(OP_END, (int32_t)readlane_u((uint32_t)end_span_of, (int)e), cp, cv);
                }
            }
            idx = uni(idx);
            ok = unib(ok);
            n_split = uni(n_split);
            above_end = idx;
            if (ok) {
                // check_remaining_edges (fill.rs:1295-1324)
                uint64_t bad = 0;
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    if ((uint32_t)c * 64u >= n_act) break;
                    const uint32_t lo = (uint32_t)c * 64u;
                    bad |= idx <= lo ? badm[c] : idx < lo + 64u ? badm[c] & ~mask_lt((int)(idx - lo)) : 0ull;
                }
                ok = bad == 0ull;
            }
            n_acts = uni(n_acts);
            status = uni(status);
            if (ok) break;
            if (attempt == 1) {
                fail(ST_INTERNAL);
                break;
            }
            // recover_from_error (fill.rs:1956-2007): rare, so one lane sorts the edges in
            // memory by the rules of sort_active_edges
            n_acts = 0;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const uint32_t i = (uint32_t)c * 64u + ul;
                if (i < n_act) {
                    AE e;
                    e.from = mk(fx[c], fy[c]);
                    e.to = mk(tx[c], ty[c]);
                    e.winding = wind_of(wm[c]);
                    e.is_merge = (wm[c] & MERGE_BIT) ? 1u : 0u;
                    e.from_id = fid[c];
                    e._pad = 0;
                    st(&g.w.act_g[i], e);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
            __builtin_amdgcn_wave_barrier();
            uint32_t sorted = 1;
            if (lane == 0)
                sorted = sort_edges_serial(g.w.act_g, g.w.act2, n_act, cp, rule) ? 1u : 0u;
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
            __builtin_amdgcn_wave_barrier();
            if (!readlane_u(sorted, 0)) {
                fail(ST_INTERNAL);
                break;
            }
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const uint32_t i = (uint32_t)c * 64u + ul;
                if (i < n_act) {
                    const AE e = ld(&g.w.act_g[i]);
                    fx[c] = e.from.x;
                    fy[c] = e.from.y;
                    tx[c] = e.to.x;
                    ty[c] = e.to.y;
                    wm[c] = ((uint32_t)e.winding & 0xffffu) | (e.is_merge ? MERGE_BIT : 0u);
                    fid[c] = e.from_id;
                }
            }
            WState w = wnew();
            for (uint32_t i = 0; i < n_act && status == ST_OK; ++i) {
                const uint32_t m = rget(wm, i);
                if (m & MERGE_BIT) w.span_index += 1;
                else wupdate(w, rule, wind_of(m));
                if (w.span_index >= (int32_t)n_spans) {
                    span_op(OP_BEGIN, w.span_index, mk(rgetf(fx, i), rgetf(fy, i)), rget(fid, i));
                    run_span_ops();
                }
            }
            if ((int64_t)n_spans > (int64_t)w.span_index + 1)
                n_spans = (uint32_t)(w.span_index + 1 > 0 ? w.span_index + 1 : 0);
            if (status != ST_OK) break;
        }
        status = uni(status);
        if (status != ST_OK) break;
        above_start = uni(above_start);
        above_end = uni(above_end);
        n_split = uni(n_split);
        merge_event = unib(merge_event);
        split_event = unib(split_event);
        wbp.number = (int32_t)uni((uint32_t)wbp.number);
        wbp.span_index = (int32_t)uni((uint32_t)wbp.span_index);
        wbp.in = rule_in(rule, wbp.number);

        // ---- process_edges_above (fill.rs:1381-1452); its span operations are queued ----
        for (uint32_t e = 0; e < n_split; ++e) {
            const uint32_t ei = readlane_u(sp_edge, (int)e);
            add_below(mk(rgetf(tx, ei), rgetf(ty, ei)), wind_of(rget(wm, ei)));
            rset(tx, ei, cp.x);
            rset(ty, ei, cp.y);
        }
        if (merge_event) {
            const uint32_t e = above_start;
            rset(fx, e, rgetf(tx, e));
            rset(fy, e, rgetf(ty, e));
            rset(wm, e, (uint32_t)MERGE_BIT);
            rset(fid, e, cv);
            above_start += 1u;
        }
        // ---- process_edges_below (fill.rs:1455-1524) ----
        // stable insertion sort by slope: a lane shift per edge that moves
        for (uint32_t i = 1; i < n_below; ++i) {
            const float v = readlane_f(b_key, (int)i);
            const uint64_t stay = ballot(ul < i && !(v < b_key));
            const uint32_t j = stay ? (uint32_t)highest_bit(stay) + 1u : 0u;
            if (j == i) continue;
            const float vx = readlane_f(b_tx, (int)i), vy = readlane_f(b_ty, (int)i);
            const uint32_t vw = readlane_u(b_w, (int)i);
            const int src = (int)(((ul - 1u) & 63u) << 2);
            const float ux = perm(b_tx, src), uy = perm(b_ty, src), uk = perm(b_key, src);
            const uint32_t uw = perm(b_w, src);
            const bool mv = ul > j && ul <= i, at = ul == j;
            b_tx = at ? vx : mv ? ux : b_tx;
            b_ty = at ? vy : mv ? uy : b_ty;
            b_key = at ? v : mv ? uk : b_key;
            b_w = at ? vw : mv ? uw : b_w;
        }
        // handle_coincident_edges_below (fill.rs:2016-2106), from the last pair down; a
        // merge changes the pair after it, so the pairs are looked at again as it goes
        if (n_below >= 2u) {
            uint32_t kk = n_below - 1u;
            while (kk > 0u && status == ST_OK) {
                const float nb = perm(b_key, (int)(((ul + 1u) & 63u) << 2));
                const float inv = ffabs(1.0f / b_key - 1.0f / nb);
                const bool flat = ffabs(b_key) <= 1.0f;
                const bool close = (flat & (ffabs(b_key - nb) < 0.00005f)) |
                                   (!flat & (inv < 0.00005f));
                const uint64_t m = ballot(close & (ul < kk) & (ul + 1u < n_below));
                if (!m) break;
                const uint32_t a = (uint32_t)highest_bit(m), b = a + 1u;
                const vec2 a_to = readlane_v(mk(b_tx, b_ty), (int)a);
                const vec2 b_to = readlane_v(mk(b_tx, b_ty), (int)b);
                const int cmp = cmp_pos(a_to, b_to);
                const uint32_t lower = cmp < 0 ? b : a, upper = cmp < 0 ? a : b;
                const int32_t lw = wind_of(readlane_u(b_w, (int)lower));
                const int32_t uw = (int16_t)(wind_of(readlane_u(b_w, (int)upper)) + lw);
                const vec2 split_point = cmp < 0 ? a_to : b_to;
                const vec2 lower_to = cmp < 0 ? b_to : a_to;
                b_w = ul == upper ? (uint32_t)uw : b_w;
                const int src = (int)(((ul + 1u) & 63u) << 2);
                const float sx = perm(b_tx, src), sy = perm(b_ty, src), sk = perm(b_key, src);
                const uint32_t sw = perm(b_w, src);
                const bool mv = ul >= lower && ul + 1u < n_below;
                b_tx = mv ? sx : b_tx;
                b_ty = mv ? sy : b_ty;
                b_key = mv ? sk : b_key;
                b_w = mv ? sw : b_w;
                n_below = uni(n_below - 1u);
                if (cmp != 0) push_later(split_point, lower_to, lw, true);
                kk = a;
            }
        }
        WState w = wbp;
        if (split_event) {  // fill.rs:1563-1608
            if (above_start == 0u || above_start >= n_act) {
                fail(ST_INTERNAL);
                break;
            }
            const uint32_t le = above_start - 1u, re = above_start;
            const vec2 lf = mk(rgetf(fx, le), rgetf(fy, le)), rf = mk(rgetf(fx, re), rgetf(fy, re));
            if (is_after(lf, rf)) span_op(OP_BEGIN, w.span_index, lf, rget(fid, le));
            else span_op(OP_BEGIN, w.span_index + 1, rf, rget(fid, re));
            span_op(OP_RIGHT, w.span_index, cp, cv);
            span_op(OP_LEFT, w.span_index + 1, cp, cv);
        }
        for (uint32_t kk = 0; kk < n_below; ++kk) {
            if (kk > 0u && w.in) span_op(OP_BEGIN, w.span_index, cp, cv);
            wupdate(w, rule, wind_of(readlane_u(b_w, (int)kk)));
        }
        if (n_acts) run_span_ops();
        if (status != ST_OK) break;

        // ---- handle_intersections (fill.rs:1611-1846) ----
        if (crossings) {
            for (uint32_t kk = 0; kk < n_below; ++kk) {
                vec2 eto = readlane_v(mk(b_tx, b_ty), (int)kk);
                const int32_t ew = wind_of(readlane_u(b_w, (int)kk));
                const float bmin = ffmin(cp.x, eto.x), bmax = fmax_(cp.x, eto.x);
                const double bfx = cp.x, bfy = cp.y, btx = eto.x, bty = eto.y;
                const double v2x = btx - bfx, v2y = bty - bfy;
                // the smallest tb, ties to the lowest index: per lane over its own edges,
                // then over the wave
                double tb_l = 1.0;
                uint32_t i_l = NONE;
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    if ((uint32_t)c * 64u >= n_act) break;
                    const uint32_t i = (uint32_t)c * 64u + ul;
                    const bool cand =
                        (i < n_act) & !((i >= above_start) & (i < above_end)) &
                        ((wm[c] & MERGE_BIT) == 0u) & !(bmin > fmax_(fx[c], tx[c])) &
                        !(bmax < ffmin(fx[c], tx[c]));
                    if (ballot(cand)) {
                        // isect_t, without branches up to the divisions
                        const double afx = fx[c], afy = fy[c], atx = tx[c], aty = ty[c];
                        const bool apart = !(((tx[c] == eto.x) & (ty[c] == eto.y)) |
                                             ((fx[c] == cp.x) & (fy[c] == cp.y)) |
                                             ((fx[c] == eto.x) & (fy[c] == eto.y)) |
                                             ((tx[c] == cp.x) & (ty[c] == cp.y)));
                        const double v1x = atx - afx, v1y = aty - afy;
                        const double v3x = bfx - afx, v3y = bfy - afy;
                        const double cr = v1x * v2y - v1y * v2x;
                        const double sign = cr > 0.0 ? 1.0 : -1.0, abs_c = fabs(cr);
                        const double t = (v3x * v2y - v3y * v2x) * sign;
                        const double u = (v3x * v1y - v3y * v1x) * sign;
                        const bool hit =
                            cand & apart & (cr != 0.0) &
                            !((t < 0.0) | (t > abs_c) | (u < 0.0) | (u > abs_c));
                        if (ballot(hit)) {
                            const double ta = t / abs_c, tb = u / abs_c;
                            const bool best =
                                hit & (tb > 0.0) & (ta > 0.0) & (ta <= 1.0) & (tb < tb_l);
                            tb_l = best ? tb : tb_l;
                            i_l = best ? i : i_l;
                        }
                    }
                }
                uint64_t m = ballot(i_l != NONE);
                if (!m) continue;
                if (__builtin_popcountll(m) > 1) {
                    // tb is in (0, 1): as a positive double its bits order like its value
                    const uint64_t tb_bits = (uint64_t)__builtin_bit_cast(int64_t, tb_l);
                    const bool f = i_l != NONE;
                    const uint32_t hi = wave_min_u32(f ? (uint32_t)(tb_bits >> 32) : ~0u);
                    const bool f1 = f && (uint32_t)(tb_bits >> 32) == hi;
                    m = ballot(f1);
                    if (__builtin_popcountll(m) > 1) {
                        const uint32_t lo = wave_min_u32(f1 ? (uint32_t)tb_bits : ~0u);
                        const bool f2 = f1 && (uint32_t)tb_bits == lo;
                        const uint32_t mi = wave_min_u32(f2 ? i_l : NONE);
                        m = ballot(f2 && i_l == mi);
                    }
                }
                const int sl = __builtin_ctzll(m);
                const uint32_t ai = readlane_u(i_l, sl);
                const uint64_t tbb = (uint64_t)__builtin_bit_cast(int64_t, tb_l);
                const double tb = __builtin_bit_cast(
                    double, (uint64_t)readlane_u((uint32_t)tbb, sl) |
                                ((uint64_t)readlane_u((uint32_t)(tbb >> 32), sl) << 32));
                // process_intersection
                const double one_t = 1.0 - tb;
                vec2 ip = mk((float)(one_t * bfx + tb * btx), (float)(one_t * bfy + tb * bty));
                if (veq(cp, ip)) {
                    rset(fx, ai, ip.x);
                    rset(fy, ai, ip.y);
                    continue;
                }
                const vec2 a_from = mk(rgetf(fx, ai), rgetf(fy, ai));
                const vec2 a_to = mk(rgetf(tx, ai), rgetf(ty, ai));
                const int32_t aw = wind_of(rget(wm, ai));
                if (!is_after(ip, cp)) ip.y = next_up(cp.y);
                if (is_near(ip, eto)) ip = eto;
                else if (is_near(ip, a_to)) ip = a_to;
                bool flipped = false;
                if (!veq(a_to, ip) && !veq(a_from, ip)) {
                    if (is_after(a_to, ip)) {
                        push_later(ip, a_to, aw, true);
                    } else {
                        flipped = true;
                        push_later(a_to, ip, -aw, true);
                    }
                    rset(tx, ai, ip.x);
                    rset(ty, ai, ip.y);
                }
                if (!veq(eto, ip) && !veq(cp, ip)) {
                    if (is_after(eto, ip)) {
                        push_later(ip, eto, ew, true);
                    } else {
                        push_later(eto, ip, -ew, true);
                        if (flipped) push_later(ip, mk(0.0f, 0.0f), 0, false);
                    }
                    b_tx = ul == kk ? ip.x : b_tx;
                    b_ty = ul == kk ? ip.y : b_ty;
                }
            }
        }
        // ---- update_active_edges (fill.rs:1527-1561) ----
        {
            const uint32_t a = above_start, removed = above_end - a, added = n_below;
            const uint32_t n_new = n_act - removed + added;
            if (n_new > act_cap) {
                fail(MORE_SETS);
                break;
            }
            if (added > removed) {
                const uint32_t d = added - removed;  // at most 64
                for (uint32_t d1 = d; d1 > 0u;) {
                    const uint32_t by = min(d1, 63u);
                    rshift_up(fx, above_end, n_act + by, by);
                    rshift_up(fy, above_end, n_act + by, by);
                    rshift_up(tx, above_end, n_act + by, by);
                    rshift_up(ty, above_end, n_act + by, by);
                    rshift_up(wm, above_end, n_act + by, by);
                    rshift_up(fid, above_end, n_act + by, by);
                    n_act += by;
                    d1 -= by;
                }
            } else if (removed > added) {
                for (uint32_t d1 = removed - added; d1 > 0u;) {
                    const uint32_t by = min(d1, 63u);
                    rshift_down(fx, a + added, n_act, by);
                    rshift_down(fy, a + added, n_act, by);
                    rshift_down(tx, a + added, n_act, by);
                    rshift_down(ty, a + added, n_act, by);
                    rshift_down(wm, a + added, n_act, by);
                    rshift_down(fid, a + added, n_act, by);
                    n_act -= by;
                    d1 -= by;
                }
            }
            if (added) {
                const int src = (int)(((ul - a) & 63u) << 2);
                const float nx = perm(b_tx, src), ny = perm(b_ty, src);
                const uint32_t nw = perm(b_w, src) & 0xffffu;
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    if ((uint32_t)c * 64u < a + added && (uint32_t)c * 64u + 63u >= a) {
                        const uint32_t i = (uint32_t)c * 64u + ul;
                        const bool me = i >= a && i < a + added;
                        fx[c] = me ? cp.x : fx[c];
                        fy[c] = me ? cp.y : fy[c];
                        tx[c] = me ? nx : tx[c];
                        ty[c] = me ? ny : ty[c];
                        wm[c] = me ? nw : wm[c];
                        fid[c] = me ? cv : fid[c];
                    }
                }
            }
            n_act = n_new;
        }
        // ---- the event's pushes (EventQueue::insert_sorted, event_queue.rs:188-250) ----
        for (uint32_t q = 0; q < n_push; ++q) {
            if (heap_n >= heap_cap) {
                fail(MORE_ROWS);
                break;
            }
            const vec2 pos = readlane_v(mk(q_px, q_py), (int)q);
            const vec2 to = readlane_v(mk(q_tx, q_ty), (int)q);
            const uint32_t w16 = readlane_u(q_w, (int)q);
            uint64_t m = ballot(h_cnt <= level);
            while (!m) {
                ++level;
                m = ballot(h_cnt <= level);
            }
            if (level >= H.rows) {
                fail(MORE_ROWS);
                break;
            }
            const uint32_t hi = fkey(pos.y), lo = fkey(pos.x);
            const bool me = lane == __builtin_ctzll(m);
            if (me) {
                const uint32_t at = 64u * h_cnt + ul;
                H.pos[at] = make_float2(pos.x, pos.y);
                H.to[at] = make_float2(to.x, to.y);
                H.meta[at] = make_uint2(heap_seq, w16);
            }
            // an equal key keeps the entry inserted earlier
            const bool first =
                me & ((hi < h_hi) | ((hi == h_hi) & (lo < h_lo)) | (h_cnt == 0u));
            h_hi = first ? hi : h_hi;
            h_lo = first ? lo : h_lo;
            h_seq = first ? heap_seq : h_seq;
            h_row = first ? h_cnt : h_row;
            h_px = first ? pos.x : h_px;
            h_py = first ? pos.y : h_py;
            h_cnt += me ? 1u : 0u;
            heap_seq = uni(heap_seq + 1u);
            heap_n = uni(heap_n + 1u);
        }
        wave_sync();
    }
    if (status == ST_OK && !crossings && (n_act != 0u || n_spans != 0u))
        status = ST_INTERNAL;
    *out_status = status;
    *out_nv = nv;
    *out_ops = n_ops;
    if (is_retry(status)) {
        const uint64_t est = (uint64_t)nv * (uint64_t)(n_static ? n_static : 1u) /
                             (uint64_t)(cur ? cur : 1u);
        *out_hint = est > 0xffffffffull ? 0xffffffffu : (uint32_t)est;
    }
}

// ---- the spans' triangles -----------------------------------------------------------------
// AdvancedMonotoneTessellator over BasicMonotoneTessellator (monotone.rs:9-404) along one
// span's operations, by one lane.  The operations are the nodes of the stack (link_stack) and
// of the side lists (link_side; the link of a list's first node is kept in registers, as a
// span's first vertex heads both).  Every triangle takes a vertex out, so a span has fewer of
// them than operations: they wait in its operations' slots, with the counts per operation,
// until the scan has placed them.
struct TSide {
    vec2 ref, prev, last_pos;
    float cons_x;
    uint32_t head, second, tail, len;
};
struct TSpan {
    FillOp* ops;
    FillTri* tri;
    uint32_t top, pside;
    TSide side[2];
    uint32_t op, cnt;           // the current operation, its triangles so far
    uint32_t slot, slot_next;   // where the next triangle goes, and the one after
};
__device__ __forceinline__ vec2 op_pos(const FillOp* ops, uint32_t i) {
    const float2 p = *reinterpret_cast<const float2*>(&ops[i].x);
    return mk(p.x, p.y);
}
// A triangle waits in the slot of one of the span's operations, in their order: there are fewer
// triangles than operations.
__device__ __forceinline__ void t_tri(TSpan& t, uint32_t a, uint32_t b, uint32_t c) {
    if (t.slot != DEAD) {
        FillTri& d = t.tri[t.slot];
        d.a = a;
        d.b = b;
        d.c = c;
        d.op = t.op;
        d.nth = t.cnt;
        t.slot = t.slot_next;
        if (t.slot != DEAD) t.slot_next = t.ops[t.slot].next;
    }
    ++t.cnt;
}
// BasicMonotoneTessellator::vertex (monotone.rs:60-107); n: the vertex's operation.
__device__ __forceinline__ void t_basic(TSpan& t, vec2 pos, uint32_t n, uint32_t side) {
    FillOp* ops = t.ops;
    const uint32_t id = ops[n].id;
    if (side != t.pside) {
        uint32_t b = t.top;
        vec2 pb = op_pos(ops, b);
        uint32_t ib = ops[b].id;
        for (uint32_t a = ops[b].link_stack; a != DEAD;) {
            const vec2 pa = op_pos(ops, a);
            const uint32_t ia = ops[a].id, nx = ops[a].link_stack;
            if (cross2(sub(pa, pb), sub(pos, pb)) >= 0.0f) t_tri(t, ia, ib, id);
            else t_tri(t, ib, ia, id);
            pb = pa;
            ib = ia;
            a = nx;
        }
        ops[t.top].link_stack = DEAD;
    } else {
        uint32_t lp = t.top;
        vec2 pl = op_pos(ops, lp);
        uint32_t il = ops[lp].id, head = ops[lp].link_stack;
        while (head != DEAD) {
            const vec2 ph = op_pos(ops, head);
            const uint32_t ih = ops[head].id;
            const vec2 na = side == 1u ? ph : pl, nb = side == 1u ? pl : ph;
            const float c = cross2(sub(pos, nb), sub(na, nb));
            if (!(c >= 0.0f)) break;
            if (side == 1u) t_tri(t, il, ih, id);
            else t_tri(t, ih, il, id);
            lp = head;
            pl = ph;
            il = ih;
            head = ops[head].link_stack;
        }
        t.top = lp;
    }
    ops[n].link_stack = t.top;
    t.top = n;
    t.pside = side;
}
// flush_side (monotone.rs:356-398): true when the side's last vertex goes to the basic
// tessellator.  Each level of the binary tree walks the list and drops every second node.
template <uint32_t SIDE>
__device__ __forceinline__ bool t_flush(TSpan& t) {
    TSide& e = t.side[SIDE];
    FillOp* ops = t.ops;
    const uint32_t len = e.len;
    if (len < 2u) return false;
    const uint32_t head = e.head, id0 = ops[head].id;
    uint32_t second = e.second;
    for (uint32_t step = 1u; step * 2u < len; step *= 2u) {
        const uint32_t imax = (len - 1u) / (2u * step);
        uint32_t a = head, ia = id0;
        for (uint32_t i = 0; i < imax; ++i) {
            const uint32_t b = a == head ? second : ops[a].link_side;
            const uint32_t l = ops[b].link_side;
            const uint32_t ib = ops[b].id, il = ops[l].id;
            if (SIDE == 1u) t_tri(t, ib, ia, il);
            else t_tri(t, ia, ib, il);
            if (a == head) second = l;
            else ops[a].link_side = l;
            a = l;
            ia = il;
        }
        if (imax * 2u * step + step < len) {
            const uint32_t c = a == head ? second : ops[a].link_side, ic = ops[c].id;
            if (SIDE == 1u) t_tri(t, id0, ic, ia);
            else t_tri(t, id0, ia, ic);
        }
    }
    e.head = e.tail;
    e.len = 1u;
    e.prev = e.last_pos;
    e.ref = e.last_pos;
    return true;
}
template <uint32_t SIDE>
__device__ __forceinline__ void t_vertex(TSpan& t, vec2 pos, uint32_t n) {
    TSide& se = t.side[SIDE];
    TSide& op = t.side[1u - SIDE];
    if (SIDE == 0u) {
        se.ref.x = ffmax(se.ref.x, pos.x);
        se.cons_x = ffmax(se.cons_x, se.ref.x);
    } else {
        se.ref.x = ffmin(se.ref.x, pos.x);
        se.cons_x = ffmin(se.cons_x, se.ref.x);
    }
    const float dx = t.side[1].cons_x - t.side[0].cons_x;
    const float dy = pos.y - se.ref.y;
    const bool close = dx < dy * 0.1f;
    bool outward = false;
    if (!close && se.len >= 2u) {
        const float sign = SIDE == 0u ? 1.0f : -1.0f;
        outward = cross2(sub(se.prev, se.last_pos), sub(pos, se.last_pos)) * sign < 0.0f;
    }
    if (outward || close) {
        if (pos_after(se.last_pos, op.last_pos)) {
            if (t_flush<1u - SIDE>(t)) {
                t_basic(t, op.last_pos, op.tail, 1u - SIDE);
                se.cons_x = se.ref.x;
            }
        }
        if (t_flush<SIDE>(t)) {
            t_basic(t, se.last_pos, se.tail, SIDE);
            op.cons_x = op.ref.x;
        }
    }
    // SideEvents::push
    if (se.len == 1u) se.second = n;
    else t.ops[se.tail].link_side = n;
    se.tail = n;
    se.len += 1u;
    se.prev = se.last_pos;
    se.last_pos = pos;
}
__device__ void t_span(FillOp* ops, FillTri* tri, uint32_t first) {
    TSpan t;
    t.ops = ops;
    t.tri = tri;
    t.slot = first;
    t.slot_next = ops[first].next;
    t.top = first;
    t.pside = 0;
    const vec2 p0 = op_pos(ops, first);
    ops[first].link_stack = DEAD;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        TSide& e = t.side[k];
        e.ref = e.prev = e.last_pos = p0;
        e.cons_x = p0.x;
        e.head = e.tail = first;
        e.second = DEAD;
        e.len = 1;
    }
    for (uint32_t n = ops[first].next; n != DEAD;) {
        const float4 r = *reinterpret_cast<const float4*>(&ops[n]);
        const vec2 pos = mk(r.x, r.y);
        const uint32_t kind = f2u(r.w), next = ops[n].next;
        t.op = n;
        t.cnt = 0;
        if (kind == OP_LEFT) {
            t_vertex<0u>(t, pos, n);
        } else if (kind == OP_RIGHT) {
            t_vertex<1u>(t, pos, n);
        } else {
            // AdvancedMonotoneTessellator::end (monotone.rs:337-353)
            const bool ha = t_flush<0u>(t);
            const bool hb = t_flush<1u>(t);
            const bool b_first = hb && (!ha || pos_after(t.side[0].last_pos, t.side[1].last_pos));
            if (b_first) t_basic(t, t.side[1].last_pos, t.side[1].tail, 1u);
            if (ha) t_basic(t, t.side[0].last_pos, t.side[0].tail, 0u);
            if (hb && !b_first) t_basic(t, t.side[1].last_pos, t.side[1].tail, 1u);
            t_basic(t, pos, n, 1u - t.pside);
        }
        ops[n].tris = t.cnt;
        n = next;
    }
    for (uint32_t q = t.slot; q != DEAD; q = ops[q].next) tri[q].op = DEAD;
}

}  // namespace fillk

// Persistent: one wave per block, each taking paths from the launch's work counter.
template <int C>
__global__ void __launch_bounds__(WAVE) fill_reg_kernel(FillLaunch L) {
    using namespace fillk;
    __shared__ uint32_t hist[256];
    extern __shared__ __align__(16) uint8_t reg_lds[];
    Cols H;
    H.rows = L.heap_rows;
    H.pos = reinterpret_cast<float2*>(reg_lds);
    H.to = H.pos + 64u * H.rows;
    H.meta = reinterpret_cast<uint2*>(H.to + 64u * H.rows);
    uint8_t* work = L.work + (size_t)blockIdx.x * L.work_stride;
    uint32_t k = readlane_u(atomicAdd(L.work_counter, lane_id() == 0 ? 1u : 0u), 0);
    while (k < L.n_list) {
        const uint32_t path = L.path_list[k];
        uint32_t st = 0, nv = 0, n_ops = 0, hint = 0;
        reg_sweep<C>(L, path, k, work, H, hist, &st, &nv, &n_ops, &hint);
        if (lane_id() == 0) {
            L.path_status[path] = st;
            L.path_nv[path] = st == 0 ? nv : 0u;
            L.path_ni[path] = 0u;  // until the triangles are counted
            L.path_ops[path] = n_ops;
            L.path_round[path] = L.round;
            if (L.path_hint) L.path_hint[path] = is_retry(st) ? hint : 0u;
        }
        k = readlane_u(atomicAdd(L.work_counter, lane_id() == 0 ? 1u : 0u), 0);
    }
}

// Lane per operation of a path (blockIdx.x: the path, blockIdx.y: a slice of its log); the
// ones that begin a span walk it, once: counting first and walking again for the triangles took
// 1,000 glyphs 237 us, 161 us so, bound by the instructions along the longest span.
__global__ void __launch_bounds__(256) fill_tess_kernel(FillLaunch L) {
    using namespace fillk;
    const uint32_t k = blockIdx.x;
    const uint32_t path = L.path_list[k];
    if (L.path_status[path] != 0u) return;
    FillOp* ops = L.ops + L.stage_t_off[k];
    FillTri* tri = L.op_tris + L.stage_t_off[k];
    const uint32_t n = L.path_ops[path];
    for (uint32_t i = blockIdx.y * 256u + threadIdx.x; i < n; i += gridDim.y * 256u)
        if (ops[i].kind == OP_BEGIN) t_span(ops, tri, i);
}

// Lane per slot: the triangles to their places, in the operations' order.
__global__ void __launch_bounds__(256) fill_tess_place_kernel(FillLaunch L) {
    using namespace fillk;
    const uint32_t k = blockIdx.x;
    const uint32_t path = L.path_list[k];
    if (L.path_status[path] != 0u) return;
    const FillOp* ops = L.ops + L.stage_t_off[k];
    const FillTri* tri = L.op_tris + L.stage_t_off[k];
    uint32_t* out = L.stage_t + 3ull * L.stage_t_off[k];
    const uint32_t n = L.path_ops[path];
    for (uint32_t i = blockIdx.y * 256u + threadIdx.x; i < n; i += gridDim.y * 256u) {
        const FillTri t = tri[i];
        if (t.op == DEAD) continue;
        uint32_t* d = out + 3ull * (ops[t.op].tris + t.nth);
        d[0] = t.a;
        d[1] = t.b;
        d[2] = t.c;
    }
}

// Wave per path: the operations' triangle counts become offsets in log order.
__global__ void __launch_bounds__(WAVE) fill_tess_scan_kernel(FillLaunch L) {
    using namespace fillk;
    const uint32_t k = blockIdx.x;
    const uint32_t path = L.path_list[k];
    const int l = lane_id();
    if (L.path_status[path] != 0u) return;
    FillOp* ops = L.ops + L.stage_t_off[k];
    const uint32_t tcap = (uint32_t)(L.stage_t_off[k + 1] - L.stage_t_off[k]);
    const uint32_t n = L.path_ops[path];
    uint32_t run = 0;
    for (uint32_t b = 0; b < n; b += 256u) {
        uint32_t c[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t i = b + 64u * (uint32_t)q + (uint32_t)l;
            c[q] = i < n ? ops[i].tris : 0u;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t i = b + 64u * (uint32_t)q + (uint32_t)l;
            const uint32_t incl = incl_scan(c[q]);
            if (i < n) ops[i].tris = run + incl - c[q];
            run += readlane_u(incl, WAVE - 1);
        }
    }
    if (l == 0) {
        const bool fits = run <= tcap;
        L.path_ni[path] = fits ? 3u * run : 0u;
        if (!fits) {
            L.path_nv[path] = 0u;
            L.path_status[path] = ST_RETRY;
            if (L.path_hint) L.path_hint[path] = run;
        }
    }
}

}  // namespace lyg

extern "C" {

// Resident waves per CU (0: it cannot launch).
int lyg_fill_reg_occupancy(uint32_t chunks, uint32_t rows) {
    int nb = 0;
    const size_t lds = lyg::fillk::cols_bytes(rows);
    const hipError_t e =
        chunks == 2 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, lyg::fill_reg_kernel<2>,
                                                                   lyg::WAVE, lds)
        : chunks == 5 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, lyg::fill_reg_kernel<5>,
                                                                     lyg::WAVE, lds)
                      : hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, lyg::fill_reg_kernel<16>,
                                                                     lyg::WAVE, lds);
    return e == hipSuccess ? nb : 0;
}
// The sweep of L's paths (L->reg_chunks register sets of 64 active edges) and its triangles.
hipError_t lyg_launch_fill_reg(const lyg::FillLaunch* L, int grid, hipStream_t s) {
    if (L->n_list == 0) return hipSuccess;
    const size_t lds = lyg::fillk::cols_bytes(L->heap_rows);
    if (L->reg_chunks == 2)
        hipLaunchKernelGGL(lyg::fill_reg_kernel<2>, dim3(grid), dim3(lyg::WAVE), lds, s, *L);
    else if (L->reg_chunks == 5)
        hipLaunchKernelGGL(lyg::fill_reg_kernel<5>, dim3(grid), dim3(lyg::WAVE), lds, s, *L);
    else if (L->reg_chunks == 16)
        hipLaunchKernelGGL(lyg::fill_reg_kernel<16>, dim3(grid), dim3(lyg::WAVE), lds, s, *L);
    else
        return hipErrorInvalidValue;
    // enough blocks for a launch of few paths to spread over the GPU
    const uint32_t slices = L->n_list >= 512u ? 4u : L->n_list >= 32u ? 16u : 64u;
    hipLaunchKernelGGL(lyg::fill_tess_kernel, dim3(L->n_list, slices), dim3(256), 0, s, *L);
    hipLaunchKernelGGL(lyg::fill_tess_scan_kernel, dim3(L->n_list), dim3(lyg::WAVE), 0, s, *L);
    hipLaunchKernelGGL(lyg::fill_tess_place_kernel, dim3(L->n_list, slices), dim3(256), 0, s, *L);
    return hipGetLastError();
}

}  // extern "C"
