// Fill tessellation for gfx950: one wave per path, sweep-line semantics of lyon's
// FillTessellator (crates/tessellation/src/fill.rs, event_queue.rs).  This is the sweep over
// arrays, for the paths that outgrow the registers of fill_reg.hip, with the kernels that
// size and copy both.
//
// The filled region must equal lyon's on the same input, including its snapping of
// vertices onto edges passing within tolerance/2, its f64 intersection points and its
// coincident-edge merging, so the event processing follows the reference's rules step
// for step (each function cites the lines it agrees with).  The machinery around it is
// built for the GPU:
//   * events are generated by one pass over the path (curves flattened after being
//     swapped downwards, as event_queue.rs:758-900) and ordered by a stable wave-wide
//     LSD radix sort on a 64-bit (y, x) key instead of a linked-list merge sort;
//   * events created during the sweep (intersections, split remainders) go into a
//     64-ary min-heap instead of a sorted linked list with linear insertion;
//   * the O(active edges) loops — locating the current point among the active edges
//     and searching the closest intersection for every new edge — run on all 64 lanes;
//   * each monotone span runs lyon's monotone tessellator (side chains + stack) with its
//     lists in a per-wave node pool, so the triangle set is lyon's; only the order of the
//     triangles in the index buffer differs.
// The sweep state is held redundantly by every lane (uniform control flow); stores to
// shared arrays are done by lane 0.
//
// Output: per path, vertices and triangles (path-local ids) go to a staging area sized by
// the host; a copy kernel moves them to the final arrays at scan offsets.
#include <hip/hip_runtime.h>

#include "lyg_math.h"
#include "lyg_types.h"
#include "wave.h"
#include "fill_core.h"

namespace lyg {

// One path on one wave.  Returns the status; nv/nt are the vertex/triangle counts.
// On a retry status, *out_hint estimates the vertices the path needs: the vertices written
// so far scaled by the fraction of the path's events already swept.
__device__ __forceinline__ void fill_one_path(const FillLaunch& L, uint32_t path, uint32_t k, uint8_t* work,
                              uint8_t* hot, uint32_t* hist, uint32_t* out_status,
                              uint32_t* out_nv, uint32_t* out_nt, uint32_t* out_hint) {
    using namespace fillk;
    Sweep s;
    s.lane = lane_id();
    s.lds_only = false;
    carve(work, hot, L.hot_bytes, L.caps, s.w);
    const lyg_fill_options o = L.opts[L.opts_stride ? path : 0];
    s.rule = o.fill_rule;
    s.no_isect = o.handle_intersections == 0;
    s.tol = o.tolerance * 0.5f;
    s.out_v = reinterpret_cast<float2*>(L.stage_v) + L.stage_v_off[k];
    s.vcap = (uint32_t)(L.stage_v_off[k + 1] - L.stage_v_off[k]);
    s.out_t = L.stage_t + 3ull * L.stage_t_off[k];
    s.tcap = (uint32_t)(L.stage_t_off[k + 1] - L.stage_t_off[k]);
    s.nv = s.nt = 0;
    s.status = ST_OK;
    s.n_act = s.n_spans = s.n_below = 0;
    s.n_nodes = 0;
    s.free_head = NODE_NONE;
    s.spans_dirty = false;
    s.heap_n = s.heap_seq = 0;
    *out_nv = 0;
    *out_nt = 0;
    // tessellate_impl (fill.rs:755-759)
    if (!(o.tolerance > 0.0f)) {
        *out_status = ST_TOLERANCE_NAN;
        return;
    }
    const bool horiz = o.sweep_orientation == LYG_ORIENT_HORIZONTAL;
    const uint32_t made = make_events(s, L.in, path, o, hist);
    if (made != ST_OK) {
        *out_status = made;
        return;
    }
    // The sorted static events are read through a ring of 32 in the radix histogram's LDS
    // (idle once the sort is done): one wave-wide refill loads 32 keys and indices and
    // gathers their events, instead of two dependent global loads per event.
    struct RingEv {
        uint64_t key;
        Ev ev;
    };
    constexpr uint32_t RING = 256u * sizeof(uint32_t) / sizeof(RingEv);
    RingEv* ring = reinterpret_cast<RingEv*>(hist);
    uint32_t ring_base = 0, ring_end = 0;  // the ring holds static events [ring_base, ring_end)
    auto ring_at = [&](uint32_t i) -> const RingEv& {  // i is wave-uniform, < n_static
        if (i >= ring_end) {
            __builtin_amdgcn_wave_barrier();
            const uint32_t j = i + (uint32_t)s.lane;
            if ((uint32_t)s.lane < RING && j < s.n_static) {
                RingEv r;
                r.key = s.w.key_a[j];
                r.ev = s.w.ev[s.w.idx_a[j]];
                ring[s.lane] = r;
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
            __builtin_amdgcn_wave_barrier();
            ring_base = i;
            ring_end = i + RING < s.n_static ? i + RING : s.n_static;
        }
        return ring[i - ring_base];
    };
    // ---- sweep (tessellator_loop, fill.rs:836-867) ----
    s.cur = 0;
    while ((s.cur < s.n_static || s.heap_n > 0) && s.status == ST_OK) {
        uint64_t ks = s.cur < s.n_static ? ring_at(s.cur).key : ~0ull;
        uint64_t kh = s.heap_n > 0 ? s.w.heap[0].key : ~0ull;
        uint64_t key = ks < kh ? ks : kh;
        vec2 pos = ks <= kh ? ring_at(s.cur).ev.pos : s.w.heap[0].ev.pos;
        s.cp = pos;
        s.cv = add_vertex(s, horiz ? mk(pos.y, -pos.x) : pos);  // fill.rs:890-894
        // initialize_events: edges below from every event at this position
        while (s.cur < s.n_static && ring_at(s.cur).key == key) {
            Ev e = ring_at(s.cur).ev;
            s.cur++;
            if (e.is_edge) {
                if (s.n_below >= s.w.below_cap &&
                    !migrate(s, s.w.below, s.w.below_cap, s.w.below_g, s.w.below_gcap, s.n_below)) {
                    fail(s, ST_RETRY);
                    break;
                }
                put(s, s.w.below, s.n_below, PE{e.to, slope(sub(e.to, s.cp)), e.winding});
                s.n_below += 1;
            }
        }
        while (s.heap_n > 0 && s.w.heap[0].key == key && s.status == ST_OK) {
            Heap h = heap_pop(s);
            if (h.ev.is_edge) {
                if (s.n_below >= s.w.below_cap &&
                    !migrate(s, s.w.below, s.w.below_cap, s.w.below_g, s.w.below_gcap, s.n_below)) {
                    fail(s, ST_RETRY);
                    break;
                }
                put(s, s.w.below, s.n_below, PE{h.ev.to, slope(sub(h.ev.to, s.cp)), h.ev.winding});
                s.n_below += 1;
            }
        }
        if (s.status != ST_OK) break;
        // process_events; on an order error recover and try once more (fill.rs:855-863)
        for (int attempt = 0; attempt < 2; ++attempt) {
            if (process_events(s)) break;
            if (attempt == 0) recover_from_error(s);
            else fail(s, ST_INTERNAL);
        }
    }
    if (s.status == ST_OK && s.no_isect && (s.n_act != 0 || s.n_spans != 0)) fail(s, ST_INTERNAL);
    *out_status = s.status;
    *out_nv = s.nv;
    *out_nt = s.nt;
    if (s.status == ST_RETRY) {
        const uint64_t est = (uint64_t)s.nv * (uint64_t)(s.n_static ? s.n_static : 1) /
                             (uint64_t)(s.cur ? s.cur : 1);
        *out_hint = est > 0xffffffffull ? 0xffffffffu : (uint32_t)est;
    }
}

static constexpr int FILL_MAX_WAVES_PER_BLOCK = 4;

// Persistent sweep: L.waves_per_block waves per block, each taking paths from the work
// counter; per wave, L.hot_bytes of the block's dynamic LDS and L.work_stride bytes of
// global working memory.
__global__ void __launch_bounds__(WAVE* FILL_MAX_WAVES_PER_BLOCK) fill_sweep_kernel(FillLaunch L) {
    __shared__ uint32_t hist_all[FILL_MAX_WAVES_PER_BLOCK][256];
    extern __shared__ __align__(16) uint8_t fill_lds[];
    const int w = threadIdx.x / WAVE;
    const uint32_t wave_slot = blockIdx.x * L.waves_per_block + w;
    uint8_t* work = L.work + (size_t)wave_slot * L.work_stride;
    uint8_t* hot = L.hot_bytes ? fill_lds + (size_t)w * L.hot_bytes : nullptr;
    uint32_t* hist = hist_all[w];
    uint32_t k = readlane_u(atomicAdd(L.work_counter, lane_id() == 0 ? 1u : 0u), 0);
    while (k < L.n_list) {
        const uint32_t path = L.path_list ? L.path_list[k] : k;
        if (L.only_retry && !fillk::is_retry(L.path_status[path])) {
            k = readlane_u(atomicAdd(L.work_counter, lane_id() == 0 ? 1u : 0u), 0);
            continue;
        }
        uint32_t st = 0, nv = 0, nt = 0, hint = 0;
        fill_one_path(L, path, k, work, hot, hist, &st, &nv, &nt, &hint);
        uint32_t* ds = L.path_status + path;
        uint32_t* dv = L.path_nv + path;
        uint32_t* dt = L.path_ni + path;
        uint32_t* dr = L.path_round + path;
        if (lane_id() == 0) {
            *ds = st;
            *dv = st == 0 ? nv : 0u;
            *dt = st == 0 ? 3u * nt : 0u;
            *dr = L.round;
            if (L.path_hint) L.path_hint[path] = st == fillk::ST_RETRY ? hint : 0u;
        }
        k = readlane_u(atomicAdd(L.work_counter, lane_id() == 0 ? 1u : 0u), 0);
    }
}

// a[list[k]] = v for the k < m paths of a round (their status until a wave sweeps them).
__global__ void fill_list_u32_kernel(uint32_t* a, const uint32_t* list, uint32_t m,
                                     uint32_t v) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < m) a[list[k]] = v;
}

// Copies each path's staged vertices and triangles to the final arrays, turning the
// path-local vertex ids into absolute ids (vertex_offset + path offset + local id).
__global__ void fill_copy_kernel(FillLaunch L) {
    const uint32_t k = blockIdx.x;
    if (k >= L.n_list) return;
    const uint32_t path = L.path_list ? L.path_list[k] : k;
    if (L.path_status[path] != 0 || L.path_round[path] != L.round) return;
    // the differences of the offsets are the path's counts even when the 32-bit scan wraps
    const uint32_t nv = L.vtx_off[path + 1] - L.vtx_off[path];
    const uint32_t ni = L.idx_off[path + 1] - L.idx_off[path];
    if ((uint64_t)L.vtx_off[path] + nv > L.vertex_capacity ||
        (uint64_t)L.idx_off[path] + ni > L.index_capacity)
        return;
    const float2* sv = reinterpret_cast<const float2*>(L.stage_v) + L.stage_v_off[k];
    const uint32_t* st = L.stage_t + 3ull * L.stage_t_off[k];
    float2* dv = reinterpret_cast<float2*>(L.out_vertices) + L.vtx_off[path];
    uint32_t* di = L.out_indices + L.idx_off[path];
    const uint32_t base = L.vertex_offset + (L.local_ids ? 0u : L.vtx_off[path]);
    for (uint32_t i = threadIdx.x; i < nv; i += blockDim.x) dv[i] = sv[i];
    for (uint32_t i = threadIdx.x; i < ni; i += blockDim.x) di[i] = st[i] + base;
}

// The callers' per-path statuses from the sweep's: a path that outgrew its room
// (retry) reports LYG_ERR_NO_SPACE, one that no wave swept LYG_ERR_INTERNAL.
__global__ void fill_status_out_kernel(const uint32_t* st, uint32_t* out, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t v = st[i];
    out[i] = fillk::is_retry(v) ? (uint32_t)LYG_ERR_NO_SPACE
                                : v == 0xffffffffu ? (uint32_t)LYG_ERR_INTERNAL : v;
}

// What sizes a path's first sweep, by a wave per path with a lane per verb:
//   * an upper bound of its events: flattened edges (the swapped-curve Wang counts) plus one
//     vertex event per edge, plus the closing edges;
//   * the sum of its segments' degrees, which a horizontal line crosses at most that often (the
//     host takes half of them for active edges: combs of more than 1,024 verbs, where that
//     decides between registers and arrays, are counted, or they outgrow the registers and
//     are swept twice: a comb of 1,500 edges 47 ms, 34 ms so);
//   * an estimate of its self-intersections, which its output and its pending events grow with
//     and the event bound does not see.  Two segments can only cross if their boxes (of the
//     control points, padded by the tolerance: the flattened edges lie within) overlap; the
//     estimate counts one crossing per overlapping pair of non-consecutive segments and one per
//     cubic (its possible loop).  For polygons this is an upper bound (two line segments cross
//     at most once); for curves it is a typical count rather than the worst case (a cubic pair
//     may cross up to 9 times, most overlapping pairs do not cross at all), and a path that
//     outgrows it is swept again with more room.  Paths with more than INTER_MAX_VERBS verbs
//     get 0 (their first attempt is sized from the events).
// CAP: the boxes one block's LDS holds.  The first launch takes every path, and raises `more`
// for those with more verbs than its boxes, up to INTER_MAX_VERBS; the second (over > 0) counts
// the pairs of those with more than `over`.  1,000 glyphs: 120 us when a thread walked a path,
// once for the bound and once for boxes in memory, 13 us so.
static constexpr uint32_t INTER_MAX_VERBS = 4096, INTER_FEW_VERBS = 1024;

// The most segments that cross one sweep line, by their boxes (padded by `pad`), to within those
// that begin or end in the same 1,024th of the path's extent.
static constexpr uint32_t CROSS_BINS = 1024;
__device__ __forceinline__ uint32_t segments_crossed(const float4* boxes, uint32_t nv, float pad,
                                                     bool horizontal, int32_t* bins) {
    const uint32_t l = (uint32_t)lane_id();
    auto top = [&](const float4& b) { return (horizontal ? b.x : b.y) + pad; };
    auto bottom = [&](const float4& b) { return (horizontal ? b.z : b.w) - pad; };
    float lo = INFINITY, hi = -INFINITY;
    for (uint32_t i = l; i < nv; i += WAVE) {
        lo = ffmin(lo, top(boxes[i]));
        hi = ffmax(hi, bottom(boxes[i]));
    }
    for (int d = 1; d < WAVE; d <<= 1) {
        lo = ffmin(lo, u2f(shfl_u(f2u(lo), (int)l ^ d)));
        hi = ffmax(hi, u2f(shfl_u(f2u(hi), (int)l ^ d)));
    }
    for (uint32_t i = l; i < CROSS_BINS; i += WAVE) bins[i] = 0;
    wave_sync();
    const float scale = (float)CROSS_BINS / (hi - lo);
    auto bin = [&](float y) {
        const float k = (y - lo) * scale;
        return k >= 1.0f ? (k < (float)CROSS_BINS ? (uint32_t)k : CROSS_BINS - 1u) : 0u;
    };
    for (uint32_t i = l; i < nv; i += WAVE) {
        const float t = top(boxes[i]), b = bottom(boxes[i]);
        if (!(t <= b)) continue;
        atomicAdd(&bins[bin(t)], 1);
        const uint32_t after = bin(b) + 1u;
        if (after < CROSS_BINS) atomicAdd(&bins[after], -1);
    }
    wave_sync();
    constexpr uint32_t PER = CROSS_BINS / WAVE;
    int32_t sum = 0, most = 0;
    for (uint32_t k = 0; k < PER; ++k) {
        sum += bins[l * PER + k];
        most = sum > most ? sum : most;
    }
    const int32_t before = (int32_t)incl_scan((uint32_t)sum) - sum;
    const int32_t here = before + most;  // (before alone is the last bin's of the lane before)
    return readlane_u(incl_max_u32(here > 0 ? (uint32_t)here : 0u), WAVE - 1);
}

template <uint32_t CAP>
__global__ void __launch_bounds__(WAVE) fill_measure_kernel(FillLaunch L, uint32_t over,
                                                            uint32_t* bound, uint32_t* degree,
                                                            uint32_t* inter, uint32_t* more) {
    __shared__ float4 boxes[CAP];
    const uint32_t path = blockIdx.x;
    const int l = lane_id();
    const uint32_t vb = L.in.verb_off[path], nv = L.in.verb_off[path + 1] - vb;
    if (over && (nv <= over || nv > CAP)) return;
    const lyg_fill_options o = L.opts[L.opts_stride ? path : 0];
    const uint32_t pb = L.in.point_off[path], npts = L.in.point_off[path + 1] - pb;
    const float2* pts = reinterpret_cast<const float2*>(L.in.points) + pb;
    // the point before index i (0: none)
    auto before = [&](uint32_t i) -> vec2 {
        if (i == 0u || i > npts) return mk(0.0f, 0.0f);
        const float2 q = pts[i - 1u];
        return mk(q.x, q.y);
    };
    const float tol = o.tolerance > 0.0f ? o.tolerance : 1.0f;
    const float pad = o.tolerance > 0.0f ? o.tolerance : 0.0f;
    const bool pairs = nv <= CAP;
    uint64_t edges = 0;
    uint32_t deg = 0, acc = 0;
    // points before the chunk; 1 + the index of the last point of a Begin, Line or curve and of
    // the latest Begin; whether the verb before the chunk ends a sub-path
    uint32_t pt = 0, c_cur = 0, c_beg = 0, c_end = 0;
    for (uint32_t v0 = 0; v0 < nv; v0 += WAVE) {
        const bool in = v0 + (uint32_t)l < nv;
        const uint32_t verb = in ? (uint32_t)L.in.verbs[vb + v0 + l] : 0xffu;
        const uint32_t np = verb == LYG_VERB_CUBIC ? 3u : verb == LYG_VERB_QUADRATIC ? 2u
                          : verb <= LYG_VERB_CLOSE ? 1u : 0u;
        const uint32_t upto = pt + incl_scan(np), first = upto - np;
        const bool moves = verb <= LYG_VERB_BEGIN;  // Line, curves, Begin
        uint32_t m = incl_max_u32(moves ? upto : 0u);
        m = m > c_cur ? m : c_cur;
        uint32_t beg = incl_max_u32(verb == LYG_VERB_BEGIN ? upto : 0u);
        beg = beg > c_beg ? beg : c_beg;
        const uint32_t is_end = in && !moves ? 1u : 0u;
        const uint32_t cur_i = from_lane_before(m, c_cur);
        const bool after_end = from_lane_before(is_end, c_end) != 0u;
        const vec2 q1 = before(first + 1u), q2 = before(first + 2u), q3 = before(first + 3u);
        uint32_t d = 0;
        float4 bx = make_float4(INFINITY, INFINITY, -INFINITY, -INFINITY);
        if (in && verb != LYG_VERB_BEGIN) {
            if (over == 0u) {
                const vec2 cur = before(cur_i);
                // the swapped curve can round one count differently: +1
                if (verb == LYG_VERB_QUADRATIC) {
                    edges += (uint64_t)seg_count(quad_wang(cur, q1, q2, tol)) + 1u;
                } else if (verb == LYG_VERB_CUBIC) {
                    edges += (uint64_t)seg_count(cubic_wang(cur, q1, q2, q3, tol)) + 1u;
                } else {
                    edges += 1u;
                }
            }
            // every sub-path is closed by an edge back to its start (event_queue.rs:661-682)
            const vec2 start = before(beg);
            const vec2 cur = after_end ? start : before(first);
            const vec2 to = !moves ? start : verb == LYG_VERB_CUBIC ? q3
                          : verb == LYG_VERB_QUADRATIC ? q2 : q1;
            const vec2 c1 = verb == LYG_VERB_QUADRATIC || verb == LYG_VERB_CUBIC ? q1 : to;
            const vec2 c2 = verb == LYG_VERB_CUBIC ? q2 : to;
            d = verb == LYG_VERB_CUBIC ? 3u : verb == LYG_VERB_QUADRATIC ? 2u : 1u;
            if (moves || !(cur.x == start.x && cur.y == start.y)) {
                bx = make_float4(ffmin(ffmin(cur.x, c1.x), ffmin(c2.x, to.x)) - pad,
                                 ffmin(ffmin(cur.y, c1.y), ffmin(c2.y, to.y)) - pad,
                                 ffmax(ffmax(cur.x, c1.x), ffmax(c2.x, to.x)) + pad,
                                 ffmax(ffmax(cur.y, c1.y), ffmax(c2.y, to.y)) + pad);
                acc += verb == LYG_VERB_CUBIC ? 1u : 0u;
            }
        }
        deg = deg + d < deg ? 0xffffffffu : deg + d;
        if (pairs && in) boxes[v0 + l] = bx;
        pt = readlane_u(upto, WAVE - 1);
        c_cur = readlane_u(m, WAVE - 1);
        c_beg = readlane_u(beg, WAVE - 1);
        c_end = readlane_u(is_end, WAVE - 1);
    }
    wave_sync();
    if (pairs) {
        for (uint32_t i = (uint32_t)l; i < nv; i += WAVE) {
            const float4 a = boxes[i];
            for (uint32_t j = i + 2; j < nv; ++j) {
                const float4 b = boxes[j];
                acc += a.x > b.z || b.x > a.z || a.y > b.w || b.y > a.w ? 0u : 1u;
            }
        }
        // a lane sees at most 64 * 4096 pairs, so 32 bits hold the sum
        const uint32_t sum = readlane_u(incl_scan(acc), WAVE - 1);
        if (l == 0) inter[path] = sum > 0x7fffffffu ? 0x7fffffffu : sum;
    } else if (l == 0) {
        inter[path] = 0u;
        if (nv <= INTER_MAX_VERBS) *more = 1u;
    }
    if (over) {
        // the host's estimate is 9/16 of the degree and 16
        __shared__ int32_t bins[CROSS_BINS];
        const uint32_t most = segments_crossed(
            boxes, nv, pad, o.sweep_orientation == LYG_ORIENT_HORIZONTAL, bins);
        const uint32_t least = most > 16u ? (most - 16u) * 16u / 9u + 2u : 0u;
        if (l == 0 && least > degree[path]) degree[path] = least;
        return;
    }
    uint64_t all_edges = 0, all_deg = 0;
    for (int i = 0; i < WAVE; ++i) {
        all_edges += (uint64_t)readlane_u((uint32_t)(edges >> 32), i) << 32 |
                     readlane_u((uint32_t)edges, i);
        all_deg += readlane_u(deg, i);
    }
    if (l == 0) {
        degree[path] = all_deg > 0xffffffffull ? 0xffffffffu : (uint32_t)all_deg;
        const uint64_t bnd = 2 * all_edges + 16;
        bound[path] = bnd > 0xffffffffull ? 0xffffffffu : (uint32_t)bnd;
    }
}

}  // namespace lyg

extern "C" {

// bound, degree, inter: n each; more: set when some path's pairs are left to a second launch
// (again), which is given the same arrays.
hipError_t lyg_launch_fill_measure(const lyg::FillLaunch* L, uint32_t n, uint32_t* bound,
                                   uint32_t* degree, uint32_t* inter, uint32_t* more, int again,
                                   hipStream_t s) {
    using namespace lyg;
    if (n == 0) return hipSuccess;
    if (again)
        hipLaunchKernelGGL(fill_measure_kernel<INTER_MAX_VERBS>, dim3(n), dim3(WAVE), 0, s, *L,
                           INTER_FEW_VERBS, bound, degree, inter, more);
    else
        hipLaunchKernelGGL(fill_measure_kernel<INTER_FEW_VERBS>, dim3(n), dim3(WAVE), 0, s, *L, 0u,
                           bound, degree, inter, more);
    return hipGetLastError();
}
size_t lyg_fill_work_bytes(const lyg::fillk::FillCaps* caps, size_t hot_bytes) {
    lyg::fillk::Work w;
    return lyg::fillk::carve(nullptr, nullptr, hot_bytes, *caps, w);
}
// Resident blocks per CU of the sweep kernel for a launch shape (0 if it cannot launch).
int lyg_fill_occupancy(uint32_t waves_per_block, uint32_t hot_bytes) {
    int nb = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &nb, lyg::fill_sweep_kernel, lyg::WAVE * (int)waves_per_block,
        (size_t)waves_per_block * hot_bytes);
    return e == hipSuccess ? nb : 0;
}
hipError_t lyg_launch_fill_sweep(const lyg::FillLaunch* L, int grid, hipStream_t s) {
    if (L->waves_per_block < 1 || L->waves_per_block > lyg::FILL_MAX_WAVES_PER_BLOCK)
        return hipErrorInvalidValue;
    const size_t lds = (size_t)L->waves_per_block * L->hot_bytes;
    hipLaunchKernelGGL(lyg::fill_sweep_kernel, dim3(grid),
                       dim3(lyg::WAVE * L->waves_per_block), lds, s, *L);
    return hipGetLastError();
}
hipError_t lyg_launch_fill_list_u32(uint32_t* a, const uint32_t* list, uint32_t m, uint32_t v,
                                    hipStream_t s) {
    if (m == 0) return hipSuccess;
    hipLaunchKernelGGL(lyg::fill_list_u32_kernel, dim3((m + 255) / 256), dim3(256), 0, s, a, list,
                       m, v);
    return hipGetLastError();
}
hipError_t lyg_launch_fill_copy(const lyg::FillLaunch* L, hipStream_t s) {
    if (L->n_list == 0) return hipSuccess;
    hipLaunchKernelGGL(lyg::fill_copy_kernel, dim3(L->n_list), dim3(256), 0, s, *L);
    return hipGetLastError();
}

hipError_t lyg_launch_fill_status_out(const uint32_t* st, uint32_t* out, uint32_t n,
                                      hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(lyg::fill_status_out_kernel, dim3((n + 255) / 256), dim3(256), 0, s, st,
                       out, n);
    return hipGetLastError();
}

}  // extern "C"
