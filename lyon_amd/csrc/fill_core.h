// The fill sweep's state and steps shared by its kernels: event generation and order, and
// the sweep over arrays in memory (lyon's rules, crates/tessellation/src/fill.rs and
// event_queue.rs; each function cites the lines it agrees with).
#pragma once
#include "lyg_math.h"
#include "lyg_types.h"
#include "wave.h"

namespace lyg {

namespace fillk {

static constexpr uint32_t NONE = 0xffffffffu;

// Orders this lane's earlier global/LDS stores before the other lanes' later loads: the
// sweep arrays are written by lane 0 and read by all lanes of the same wave.  Only one wave
// touches them, so a wavefront-scope fence suffices (a wave's memory operations reach LDS
// and the vector cache in its program order; the compiler emits no wait for it).  The sweep
// over arrays keeps the workgroup scope: its flat accesses wait on every counter anyway.
template <class S>
__device__ __forceinline__ void gsync(const S& s) {
    if (s.lds_only) __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    else __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
}

enum : uint32_t {
    ST_OK = 0,
    ST_TOO_MANY_VERTICES = 1,
    ST_POSITION_NAN = 3,
    ST_TOLERANCE_NAN = 4,
    ST_INTERNAL = 5,
};

__device__ __forceinline__ int cmp_pos(vec2 a, vec2 b) {
    if (a.y > b.y) return 1;
    if (a.y < b.y) return -1;
    if (a.x > b.x) return 1;
    if (a.x < b.x) return -1;
    return 0;
}
__device__ __forceinline__ bool is_after(vec2 a, vec2 b) {
    return a.y > b.y || (a.y == b.y && a.x > b.x);
}
__device__ __forceinline__ bool is_near(vec2 a, vec2 b) { return sqlen(sub(a, b)) < 0.000000001f; }
__device__ __forceinline__ float fmax_(float a, float b) { return a > b ? a : b; }
// fill.rs:64-66
__device__ __forceinline__ float slope(vec2 v) { return v.x / ffmax(v.y, 1.17549435e-38f); }
__device__ __forceinline__ bool rule_in(uint32_t rule, int32_t w) {
    int16_t n = (int16_t)w;
    return rule == 0 ? (n % 2 != 0) : (n != 0);
}
// Order-preserving 32-bit key of an f32 (with -0 folded onto +0).
__device__ __forceinline__ uint32_t fkey(float f) {
    if (f == 0.0f) f = 0.0f;
    uint32_t u = f2u(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ uint64_t pkey(vec2 p) { return ((uint64_t)fkey(p.y) << 32) | fkey(p.x); }

struct Ev {  // an event: a position with an optional edge going down from it
    vec2 pos, to;
    int32_t winding;
    uint32_t is_edge;
};

struct AE {  // ActiveEdge (fill.rs:153-170) without the vertex-source metadata
    vec2 from, to;
    int32_t winding;
    uint32_t is_merge;
    uint32_t from_id;
    uint32_t _pad;
    __device__ float min_x() const { return ffmin(from.x, to.x); }
    __device__ float max_x() const { return fmax_(from.x, to.x); }
    // fill.rs:181-195 + LineSegment::solve_x_for_y (line.rs:56-71)
    __device__ float solve_x_for_y(float y) const {
        float dy = to.y - from.y;
        float t = dy == 0.0f ? 0.0f : (y - from.y) / dy;
        float x = from.x * (1.0f - t) + to.x * t;
        return ffmin(ffmax(x, min_x()), max_x());
    }
};

struct PE {  // PendingEdge (fill.rs:302-310)
    vec2 to;
    float sort_key;
    int32_t winding;
};

struct SideEv {  // SideEvents (monotone.rs:189-213)
    vec2 ref;        // reference_point
    float cons_x;    // conservative_reference_x
    vec2 prev;
    vec2 last_pos;   // last: MonotoneVertex
    uint32_t last_id, last_side;
    uint32_t ev_head, ev_tail, ev_len;  // events: ids, a list in the node pool
};

struct Span {  // one monotone span: AdvancedMonotoneTessellator state
    vec2 ppos;       // BasicMonotoneTessellator::previous
    uint32_t pid, pside;
    uint32_t head;   // top of the BasicMonotoneTessellator stack (node index)
    uint32_t alive;
    SideEv side[2];  // left, right
};

struct Node {  // one stack entry of a span, in the wave's node pool
    vec2 pos;
    uint32_t id;
    uint32_t side_next;  // side in bit 31, next node in bits 0-30 (0x7fffffff: none)
};
static constexpr uint32_t NODE_NONE = 0x7fffffffu;

struct Heap {  // min-heap entries: key then insertion sequence
    uint64_t key;
    uint32_t seq, _pad;
    Ev ev;
};

// Per-wave working memory, carved out of one scratch block.
struct Work {
    uint64_t* key_a;
    uint32_t* idx_a;
    uint64_t* key_b;
    uint32_t* idx_b;
    Ev* ev;
    Heap* heap;
    AE* act;
    AE* act2;
    Span* spans;
    Node* nodes;
    uint32_t* flat;      // a side's events copied out for flush_side (node_cap entries)
    PE* below;
    int32_t* vev_span;   // scan.vertex_events (span, side)
    uint32_t* vev_side;
    uint32_t* to_split;  // scan.edges_to_split
    int32_t* to_end;     // scan.spans_to_end
    uint32_t ev_cap, heap_cap, act_cap, span_cap, below_cap, node_cap;  // current capacities
    // The arrays above start in LDS when they fit; each also has a global region of the
    // worst-case capacity, where it moves when its LDS capacity overflows.
    Heap* heap_g;
    AE* act_g;
    Span* spans_g;
    Node* nodes_g;
    uint32_t* flat_g;
    PE* below_g;
    uint32_t* to_split_g;
    int32_t* to_end_g;
    uint32_t heap_gcap, act_gcap, span_gcap, below_gcap, node_gcap;
};

// LDS capacities for a per-wave budget: shares of the budget for the arrays the sweep
// touches on every event (never above the worst case).
__host__ __device__ inline FillCaps hot_caps(const FillCaps& c, size_t budget) {
    auto part = [&](double frac, size_t elem, uint32_t worst) {
        const size_t n = (size_t)(frac * (double)budget) / elem;
        return (uint32_t)(n < worst ? n : worst);
    };
    FillCaps h;
    h.ev = 0;
    h.act = part(0.26, sizeof(AE) + 8, c.act);  // + to_split, to_end entries
    h.span = part(0.30, sizeof(Span), c.span);
    h.node = part(0.22, sizeof(Node) + 4, c.node);  // + flat entry
    h.heap = part(0.12, sizeof(Heap), c.heap);
    h.below = part(0.05, sizeof(PE), c.below);
    return h;
}

// Lays out one wave's working memory: every sweep array gets a global region of its
// worst-case capacity; the arrays touched on every event also get an LDS region (of the
// hot_caps capacity) where they start, when `hot` is given.  The event arrays (read once,
// in order) are global only.  With null pointers it only measures: the return value is the
// global bytes per wave.
__host__ __device__ inline size_t carve(uint8_t* base, uint8_t* hot, size_t hot_bytes,
                                        const FillCaps& c, Work& w) {
    size_t go = 0, ho = 0;
    auto g = [&](size_t bytes) -> uint8_t* {
        uint8_t* p = base ? base + go : nullptr;
        go = (go + bytes + 255) & ~(size_t)255;
        return p;
    };
    auto h = [&](size_t bytes) -> uint8_t* {
        uint8_t* p = hot ? hot + ho : nullptr;
        ho += (bytes + 15) & ~(size_t)15;
        return p;
    };
    Work t;
    t.ev_cap = c.ev;
    t.heap_gcap = c.heap;
    t.act_gcap = c.act;
    t.span_gcap = c.span;
    t.node_gcap = c.node;
    t.below_gcap = c.below;
    t.act_g = (AE*)g(sizeof(AE) * (size_t)c.act);
    t.below_g = (PE*)g(sizeof(PE) * (size_t)c.below);
    t.to_split_g = (uint32_t*)g(4ull * c.act);
    t.to_end_g = (int32_t*)g(4ull * c.act + 16);
    t.spans_g = (Span*)g(sizeof(Span) * (size_t)c.span);
    t.nodes_g = (Node*)g(sizeof(Node) * (size_t)c.node);
    t.flat_g = (uint32_t*)g(4ull * c.node);
    t.heap_g = (Heap*)g(sizeof(Heap) * (size_t)c.heap);
    t.act2 = (AE*)g(sizeof(AE) * (size_t)c.act);
    t.key_a = (uint64_t*)g(8ull * c.ev);
    t.idx_a = (uint32_t*)g(4ull * c.ev);
    t.key_b = (uint64_t*)g(8ull * c.ev);
    t.idx_b = (uint32_t*)g(4ull * c.ev);
    t.ev = (Ev*)g(sizeof(Ev) * (size_t)c.ev);
    const FillCaps hc = hot_caps(c, hot_bytes);
    // scan lists are tiny: always in LDS when there is LDS
    const bool use_hot = hot_bytes >= 256;
    t.vev_span = use_hot ? (int32_t*)h(4 * 8) : (int32_t*)g(4 * 8);
    t.vev_side = use_hot ? (uint32_t*)h(4 * 8) : (uint32_t*)g(4 * 8);
    auto pick = [&](uint32_t hcap, uint32_t gcap) { return use_hot && hcap >= 8 && hcap < gcap; };
    if (pick(hc.act, c.act)) {
        t.act = (AE*)h(sizeof(AE) * (size_t)hc.act);
        t.to_split = (uint32_t*)h(4ull * hc.act);
        t.to_end = (int32_t*)h(4ull * hc.act + 16);
        t.act_cap = hc.act;
    } else {
        t.act = t.act_g;
        t.to_split = t.to_split_g;
        t.to_end = t.to_end_g;
        t.act_cap = c.act;
    }
    if (pick(hc.below, c.below)) {
        t.below = (PE*)h(sizeof(PE) * (size_t)hc.below);
        t.below_cap = hc.below;
    } else {
        t.below = t.below_g;
        t.below_cap = c.below;
    }
    if (pick(hc.span, c.span)) {
        t.spans = (Span*)h(sizeof(Span) * (size_t)hc.span);
        t.span_cap = hc.span;
    } else {
        t.spans = t.spans_g;
        t.span_cap = c.span;
    }
    if (pick(hc.node, c.node)) {
        t.nodes = (Node*)h(sizeof(Node) * (size_t)hc.node);
        t.flat = (uint32_t*)h(4ull * hc.node);
        t.node_cap = hc.node;
    } else {
        t.nodes = t.nodes_g;
        t.flat = t.flat_g;
        t.node_cap = c.node;
    }
    if (pick(hc.heap, c.heap)) {
        t.heap = (Heap*)h(sizeof(Heap) * (size_t)hc.heap);
        t.heap_cap = hc.heap;
    } else {
        t.heap = t.heap_g;
        t.heap_cap = c.heap;
    }
    w = t;
    return go + 256;
}

}  // namespace fillk

namespace fillk {

struct WState {  // WindingState (fill.rs:89-113)
    int32_t span_index;
    int32_t number;
    bool in;
};
__device__ __forceinline__ WState wnew() { return WState{-1, 0, false}; }
__device__ __forceinline__ void wupdate(WState& w, uint32_t rule, int32_t ew) {
    w.number = (int16_t)(w.number + ew);
    w.in = rule_in(rule, w.number);
    if (w.in) w.span_index += 1;
}

// All sweep state; every lane holds an identical copy.
struct Sweep {
    Work w;
    bool lds_only;  // only this wave's own memory is used (the register sweep's events)
    int lane;
    uint32_t rule;
    float tol;  // snapping threshold: options.tolerance * 0.5 (fill.rs:772-778)
    bool no_isect;
    float2* out_v;
    uint32_t vcap, nv;
    uint32_t* out_t;
    uint32_t tcap, nt;
    uint32_t status;
    uint32_t n_static, cur, heap_n, heap_seq;
    vec2 cp;
    uint32_t cv;
    uint32_t n_act, n_spans, n_below;
    uint32_t n_nodes, free_head;  // node pool: bump count and free list
    bool spans_dirty;             // a span ended since the last cleanup
    // scan results (fill.rs:116-150)
    uint32_t n_vev, n_split, n_end;
    bool merge_event, split_event, merge_split_event;
    uint32_t above_start, above_end;
    WState wbp;
};

__device__ __forceinline__ void fail(Sweep& s, uint32_t st) {
    if (s.status == ST_OK) s.status = st;
}

// ---- output ------------------------------------------------------------------------
__device__ __forceinline__ uint32_t add_vertex(Sweep& s, vec2 p) {
    uint32_t id = s.nv++;
    if (id < s.vcap) {
        if (s.lane == 0) s.out_v[id] = make_float2(p.x, p.y);
    } else {
        fail(s, ST_RETRY);
    }
    return id;
}
__device__ __forceinline__ void add_tri(Sweep& s, uint32_t a, uint32_t b, uint32_t c) {
    uint32_t t = s.nt++;
    if (t < s.tcap) {
        if (s.lane == 0) {
            s.out_t[3 * t + 0] = a;
            s.out_t[3 * t + 1] = b;
            s.out_t[3 * t + 2] = c;
        }
    } else {
        fail(s, ST_RETRY);
    }
}

// ---- lane-parallel array moves ---------------------------------------------------------
// a[from..n) -> a[from+by..n+by), top chunk first.
template <class T>
__device__ void shift_right(Sweep& s, T* a, uint32_t from, uint32_t n, uint32_t by) {
    for (int64_t hi = n; hi > (int64_t)from; hi -= WAVE) {
        int64_t lo = hi - WAVE < (int64_t)from ? (int64_t)from : hi - WAVE;
        int64_t i = lo + s.lane;
        T v;
        bool act = i < hi;
        if (act) v = ld(a + i);
        gsync(s);
        if (act) st(a + i + by, v);
        gsync(s);
    }
}
// a[from+by..n) -> a[from..n-by)
template <class T>
__device__ void shift_left(Sweep& s, T* a, uint32_t from, uint32_t n, uint32_t by) {
    for (uint32_t lo = from + by; lo < n; lo += WAVE) {
        uint32_t i = lo + s.lane;
        T v;
        bool act = i < n;
        if (act) v = ld(a + i);
        gsync(s);
        if (act) st(a + i - by, v);
        gsync(s);
    }
}
// Element copies word by word, so that array elements travel through registers (a plain
// struct assignment between two array slots goes through a private-memory temporary).
template <class T>
__device__ __forceinline__ T ld(const T* p) {
    static_assert(sizeof(T) % 4 == 0, "word-sized elements");
    uint32_t w[sizeof(T) / 4];
    const uint32_t* q = reinterpret_cast<const uint32_t*>(p);
#pragma unroll
    for (unsigned k = 0; k < sizeof(T) / 4; ++k) w[k] = q[k];
    T v;
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}
template <class T>
__device__ __forceinline__ void st(T* p, const T& v) {
    uint32_t w[sizeof(T) / 4];
    __builtin_memcpy(w, &v, sizeof(T));
    uint32_t* q = reinterpret_cast<uint32_t*>(p);
#pragma unroll
    for (unsigned k = 0; k < sizeof(T) / 4; ++k) q[k] = w[k];
}

// Lane 0 stores one element of a shared array.  The leading sync keeps every lane's
// earlier loads ahead of the store (a lane must not see a value written "after" its read),
// the trailing one makes the store visible to every lane's next load.
template <class T>
__device__ __forceinline__ void put(Sweep& s, T* a, uint32_t i, const T& v) {
    gsync(s);
    if (s.lane == 0) st(a + i, v);
    gsync(s);
}

// Lane 0 stores without the trailing sync, for sequences that never read back a slot they
// wrote (heap sifts, list walks); the sequence ends with one gsync().  The wave barrier
// keeps the store after the lanes' earlier loads of the same step.
template <class T>
__device__ __forceinline__ void put_nf(Sweep& s, T* a, uint32_t i, const T& v) {
    __builtin_amdgcn_wave_barrier();
    if (s.lane == 0) st(a + i, v);
}

// Moves an array from its LDS region to its global region (copying the `live` elements)
// when its LDS capacity is exhausted; false when it already is in global memory.
template <class T>
__device__ __forceinline__ bool migrate(Sweep& s, T*& p, uint32_t& cap, T* gp, uint32_t gcap,
                                        uint32_t live) {
    if (s.lds_only || p == gp || gcap <= cap) return false;
    for (uint32_t base = 0; base < live; base += WAVE) {
        const uint32_t i = base + s.lane;
        if (i < live) st(gp + i, ld(p + i));
    }
    gsync(s);
    p = gp;
    cap = gcap;
    return true;
}

// ---- spans: monotone triangulation ---------------------------------------------------
// Each span runs lyon's AdvancedMonotoneTessellator (monotone.rs:189-404) over its
// BasicMonotoneTessellator (monotone.rs:9-139), so a span yields the triangles lyon's
// yields.  The stack and the two side-event lists are linked lists in a per-wave node
// pool.  Triangles are written as soon as they are formed (lyon buffers a span's
// triangles until the span ends; on an error both discard the whole geometry), so only
// their order in the index buffer differs.
__device__ __forceinline__ Node node_at(const Sweep& s, uint32_t n) { return ld(&s.w.nodes[n]); }
__device__ __forceinline__ uint32_t node_next(const Node& n) { return n.side_next & NODE_NONE; }

__device__ __forceinline__ uint32_t node_alloc(Sweep& s, vec2 pos, uint32_t id, uint32_t side, uint32_t next) {
    uint32_t n;
    if (s.free_head != NODE_NONE) {
        n = s.free_head;
        s.free_head = node_next(node_at(s, n));
    } else if (s.n_nodes < s.w.node_cap && s.n_nodes < NODE_NONE) {
        n = s.n_nodes++;
    } else {
        if (s.n_nodes < NODE_NONE &&
            migrate(s, s.w.nodes, s.w.node_cap, s.w.nodes_g, s.w.node_gcap, s.n_nodes)) {
            s.w.flat = s.w.flat_g;  // flat is dead between flushes; it follows the pool
            n = s.n_nodes++;
        } else {
            fail(s, ST_RETRY);
            return NODE_NONE;
        }
    }
    Node nd{pos, id, (side << 31) | (next & NODE_NONE)};
    put(s, s.w.nodes, n, nd);
    return n;
}
__device__ __forceinline__ void node_set_next(Sweep& s, uint32_t n, uint32_t next) {
    Node nd = node_at(s, n);
    nd.side_next = (nd.side_next & 0x80000000u) | (next & NODE_NONE);
    put(s, s.w.nodes, n, nd);
}
__device__ __forceinline__ void node_free(Sweep& s, uint32_t n) {
    node_set_next(s, n, s.free_head);
    s.free_head = n;
}
// Frees the list starting at `n`, stopping before `stop`.
__device__ __forceinline__ void free_list(Sweep& s, uint32_t n, uint32_t stop) {
    uint32_t guard = 0;
    while (n != NODE_NONE && n != stop && s.status == ST_OK) {
        uint32_t next = node_next(node_at(s, n));
        node_free(s, n);
        n = next;
        if (++guard > s.w.node_gcap) fail(s, ST_INTERNAL);
    }
}
__device__ __forceinline__ float cross2(vec2 a, vec2 b) { return a.x * b.y - a.y * b.x; }

// BasicMonotoneTessellator::monotone_vertex (monotone.rs:60-107).
__device__ __forceinline__ void monotone_vertex(Sweep& s, Span& sp, vec2 pos, uint32_t id, uint32_t side) {
    if (side != sp.pside) {
        // fan the new vertex with every consecutive pair of the stack, then keep only
        // the previous vertex (always the top of the stack) under the new one
        const uint32_t top = sp.head;
        uint32_t b = top;
        uint32_t guard = 0;
        while (b != NODE_NONE && s.status == ST_OK) {
            Node nb = node_at(s, b);
            uint32_t a = node_next(nb);
            if (a == NODE_NONE) break;
            Node na = node_at(s, a);
            // the pair (a below b): triangle (a, b, new) or (b, a, new) by winding
            bool winding = cross2(sub(na.pos, nb.pos), sub(pos, nb.pos)) >= 0.0f;
            if (winding) add_tri(s, na.id, nb.id, id);
            else add_tri(s, nb.id, na.id, id);
            if (b != top) node_free(s, b);
            b = a;
            if (++guard > s.w.node_gcap) fail(s, ST_INTERNAL);
        }
        if (b != NODE_NONE && b != top) node_free(s, b);
        if (top != NODE_NONE) node_set_next(s, top, NODE_NONE);
        sp.head = top;
    } else {
        uint32_t lp = sp.head;  // last popped
        uint32_t head = NODE_NONE;
        if (lp != NODE_NONE) head = node_next(node_at(s, lp));
        uint32_t guard = 0;
        while (head != NODE_NONE && s.status == ST_OK) {
            Node na = node_at(s, lp), nb = node_at(s, head);
            if (side == 1) {
                Node t = na;
                na = nb;
                nb = t;
            }
            float c = cross2(sub(pos, nb.pos), sub(na.pos, nb.pos));
            if (!(c >= 0.0f)) break;
            add_tri(s, nb.id, na.id, id);
            node_free(s, lp);
            lp = head;
            head = node_next(node_at(s, head));
            if (++guard > s.w.node_gcap) fail(s, ST_INTERNAL);
        }
        if (lp != NODE_NONE) {
            node_set_next(s, lp, head);
            head = lp;
        }
        sp.head = head;
    }
    uint32_t n = node_alloc(s, pos, id, side, sp.head);
    if (n != NODE_NONE) sp.head = n;
    sp.ppos = pos;
    sp.pid = id;
    sp.pside = side;
}

// SideEvents::push (monotone.rs:207-212)
__device__ __forceinline__ void side_push(Sweep& s, SideEv& e, vec2 pos, uint32_t id, uint32_t side) {
    uint32_t n = node_alloc(s, pos, id, side, NODE_NONE);
    if (n == NODE_NONE) return;
    if (e.ev_tail != NODE_NONE) node_set_next(s, e.ev_tail, n);
    else e.ev_head = n;
    e.ev_tail = n;
    e.ev_len += 1;
    e.prev = e.last_pos;
    e.last_pos = pos;
    e.last_id = id;
    e.last_side = side;
}

// Triangles (ids[a], ids[b], ids[c]) for the lanes with `act`, written as one block.
__device__ __forceinline__ void add_tris_lanes(Sweep& s, bool act, uint32_t a, uint32_t b, uint32_t c) {
    uint64_t m = ballot(act);
    uint32_t cnt = (uint32_t)__builtin_popcountll(m);
    if (cnt == 0) return;
    uint32_t rank = (uint32_t)__builtin_popcountll(m & mask_lt(s.lane));
    uint32_t t = s.nt + rank;
    if (act && t < s.tcap) {
        s.out_t[3ull * t + 0] = a;
        s.out_t[3ull * t + 1] = b;
        s.out_t[3ull * t + 2] = c;
    }
    s.nt += cnt;
    if (s.nt > s.tcap) fail(s, ST_RETRY);
}

// flush_side (monotone.rs:356-398).  Returns whether a vertex must go to the basic
// tessellator (it is the side's last vertex).
__device__ __forceinline__ bool flush_side(Sweep& s, SideEv& e, uint32_t side) {
    const uint32_t len = e.ev_len;
    if (len < 2) return false;
    // the events in push order into `flat`
    {
        uint32_t n = e.ev_head;
        for (uint32_t k = 0; k < len && s.status == ST_OK; ++k) {
            if (n == NODE_NONE || k >= s.w.node_cap) {
                fail(s, ST_INTERNAL);
                break;
            }
            Node nd = node_at(s, n);
            if (s.lane == 0) s.w.flat[k] = nd.id;
            n = node_next(nd);
        }
        gsync(s);
    }
    if (s.status != ST_OK) return false;
    const uint32_t* ev = s.w.flat;
    for (uint32_t step = 1; step * 2 < len; step *= 2) {
        const uint32_t imax = (len - 1) / (2 * step);
        for (uint32_t base = 0; base < imax; base += WAVE) {
            uint32_t i = base + s.lane;
            bool act = i < imax;
            uint32_t ta = 0, tb = 0, tc = 0;
            if (act) {
                uint32_t a = i * 2 * step, b = a + step, l = b + step;
                if (side == 1) {
                    uint32_t t = a;
                    a = b;
                    b = t;
                }
                ta = ev[a];
                tb = ev[b];
                tc = ev[l];
            }
            add_tris_lanes(s, act, ta, tb, tc);
        }
        const uint32_t last_index = imax * 2 * step;
        if (last_index + step < len) {
            uint32_t b = last_index, c = last_index + step;
            if (side == 1) {
                uint32_t t = b;
                b = c;
                c = t;
            }
            add_tri(s, ev[0], ev[b], ev[c]);
        }
    }
    gsync(s);
    // events = [last] (the tail node holds the last id); prev = last; reference = last
    free_list(s, e.ev_head, e.ev_tail);
    e.ev_head = e.ev_tail;
    e.ev_len = 1;
    e.prev = e.last_pos;
    e.ref = e.last_pos;
    return true;
}

__device__ __forceinline__ bool pos_after(vec2 a, vec2 b) {
    return a.y > b.y || (a.y == b.y && a.x > b.x);
}

// AdvancedMonotoneTessellator::vertex (monotone.rs:276-335); SIDE is a template argument
// so the span's two side records stay in registers.
template <uint32_t SIDE>
__device__ __forceinline__ void adv_vertex_side(Sweep& s, Span& sp, vec2 pos, uint32_t id) {
    SideEv& se = sp.side[SIDE];
    SideEv& op = sp.side[1 - SIDE];
    if (SIDE == 0) {
        se.ref.x = ffmax(se.ref.x, pos.x);
        se.cons_x = ffmax(se.cons_x, se.ref.x);
    } else {
        se.ref.x = ffmin(se.ref.x, pos.x);
        se.cons_x = ffmin(se.cons_x, se.ref.x);
    }
    const float dx = sp.side[1].cons_x - sp.side[0].cons_x;
    const float dy = pos.y - se.ref.y;
    const bool sides_are_close = dx < dy * 0.1f;
    bool outward_turn = false;
    if (!sides_are_close && se.ev_len >= 2) {
        const float sign = SIDE == 0 ? 1.0f : -1.0f;
        outward_turn = cross2(sub(se.prev, se.last_pos), sub(pos, se.last_pos)) * sign < 0.0f;
    }
    if (outward_turn || sides_are_close) {
        const bool must_flush_opposite = pos_after(se.last_pos, op.last_pos);
        if (must_flush_opposite) {
            if (flush_side(s, op, 1 - SIDE)) {
                monotone_vertex(s, sp, op.last_pos, op.last_id, op.last_side);
                se.cons_x = se.ref.x;
            }
        }
        if (flush_side(s, se, SIDE)) {
            monotone_vertex(s, sp, se.last_pos, se.last_id, se.last_side);
            op.cons_x = op.ref.x;
        }
    }
    side_push(s, se, pos, id, SIDE);
}
__device__ __forceinline__ void adv_vertex(Sweep& s, Span& sp, vec2 pos, uint32_t id, uint32_t side) {
    if (side == 0) adv_vertex_side<0>(s, sp, pos, id);
    else adv_vertex_side<1>(s, sp, pos, id);
}

__device__ __forceinline__ void begin_span(Sweep& s, int32_t idx, vec2 pos, uint32_t id) {
    if (idx < 0 || (uint32_t)idx > s.n_spans) {
        fail(s, ST_INTERNAL);
        return;
    }
    if (s.n_spans + 1 > s.w.span_cap &&
        !migrate(s, s.w.spans, s.w.span_cap, s.w.spans_g, s.w.span_gcap, s.n_spans)) {
        fail(s, ST_RETRY);
        return;
    }
    shift_right(s, s.w.spans, (uint32_t)idx, s.n_spans, 1);
    // AdvancedMonotoneTessellator::begin (monotone.rs:248-274)
    Span sp;
    sp.ppos = pos;
    sp.pid = id;
    sp.pside = 0;
    sp.alive = 1;
    sp.head = node_alloc(s, pos, id, 0, NODE_NONE);
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) {
        SideEv& e = sp.side[k];
        e.ref = pos;
        e.cons_x = pos.x;
        e.prev = pos;
        e.last_pos = pos;
        e.last_id = id;
        e.last_side = k;
        e.ev_head = e.ev_tail = NODE_NONE;
        e.ev_len = 0;
        side_push(s, e, pos, id, k);
    }
    put(s, s.w.spans, (uint32_t)idx, sp);
    s.n_spans += 1;
}
__device__ __forceinline__ void span_vertex(Sweep& s, int32_t idx, vec2 pos, uint32_t id, uint32_t side) {
    if (idx < 0 || (uint32_t)idx >= s.n_spans) {
        fail(s, ST_INTERNAL);
        return;
    }
    Span sp = ld(&s.w.spans[idx]);
    if (!sp.alive) {
        fail(s, ST_INTERNAL);
        return;
    }
    adv_vertex(s, sp, pos, id, side);
    put(s, s.w.spans, (uint32_t)idx, sp);
}
// AdvancedMonotoneTessellator::end (monotone.rs:337-353), then the lists are released.
__device__ __forceinline__ void end_span(Sweep& s, int32_t idx, vec2 pos, uint32_t id) {
    if (idx < 0 || (uint32_t)idx >= s.n_spans) {
        fail(s, ST_INTERNAL);
        return;
    }
    Span sp = ld(&s.w.spans[idx]);
    if (!sp.alive) {  // unreachable!() in Spans::end_span (fill.rs:256-261)
        fail(s, ST_INTERNAL);
        return;
    }
    const bool ha = flush_side(s, sp.side[0], 0);
    const bool hb = flush_side(s, sp.side[1], 1);
    const SideEv& A = sp.side[0];
    const SideEv& Bv = sp.side[1];
    if (ha && !hb) {
        monotone_vertex(s, sp, A.last_pos, A.last_id, A.last_side);
    } else if (!ha && hb) {
        monotone_vertex(s, sp, Bv.last_pos, Bv.last_id, Bv.last_side);
    } else if (ha && hb) {
        if (pos_after(A.last_pos, Bv.last_pos)) {
            monotone_vertex(s, sp, Bv.last_pos, Bv.last_id, Bv.last_side);
            monotone_vertex(s, sp, sp.side[0].last_pos, sp.side[0].last_id, sp.side[0].last_side);
        } else {
            monotone_vertex(s, sp, A.last_pos, A.last_id, A.last_side);
            monotone_vertex(s, sp, sp.side[1].last_pos, sp.side[1].last_id, sp.side[1].last_side);
        }
    }
    // BasicMonotoneTessellator::end (monotone.rs:109-113)
    monotone_vertex(s, sp, pos, id, 1u - sp.pside);
    free_list(s, sp.head, NODE_NONE);
    free_list(s, sp.side[0].ev_head, NODE_NONE);
    free_list(s, sp.side[1].ev_head, NODE_NONE);
    sp.head = NODE_NONE;
    sp.alive = 0;
    put(s, s.w.spans, (uint32_t)idx, sp);
    s.spans_dirty = true;
}
// Spans::cleanup_spans (fill.rs:295-298): drops the spans that ended, keeping the order.
// Runs only after a span ended; 64 spans per step, each live span moved to its rank.
__device__ __forceinline__ void cleanup_spans(Sweep& s) {
    if (!s.spans_dirty) return;
    s.spans_dirty = false;
    uint32_t j = 0;
    for (uint32_t base = 0; base < s.n_spans; base += WAVE) {
        const uint32_t i = base + s.lane;
        Span sp;
        bool alive = false;
        if (i < s.n_spans) {
            sp = ld(&s.w.spans[i]);
            alive = sp.alive != 0;
        }
        const uint64_t m = ballot(alive);
        const uint32_t dst = j + (uint32_t)__builtin_popcountll(m & mask_lt(s.lane));
        gsync(s);  // every read of this chunk before any write (dst <= i)
        if (alive && dst != i) st(&s.w.spans[dst], sp);
        gsync(s);
        j += (uint32_t)__builtin_popcountll(m);
    }
    s.n_spans = j;
}

// ---- event heap ----------------------------------------------------------------------
__device__ __forceinline__ bool heap_less(const Heap& a, const Heap& b) {
    return a.key < b.key || (a.key == b.key && a.seq < b.seq);
}
// 64-ary heap: a node's children are the 64 slots 64 i + 1 ... 64 i + 64, so a sift-down
// level is one lane-parallel load of the children's (key, seq) and a wave minimum, and a
// heap of n events is log64(n) levels deep.  The order of the pops is the (key, seq)
// order whatever the arity.
__device__ __forceinline__ uint32_t heap_min_child(const Sweep& s, uint32_t first) {
    const uint32_t c = first + (uint32_t)s.lane;
    const bool valid = c < s.heap_n;
    uint32_t lo = ~0u, hi = ~0u, sq = ~0u;
    if (valid) {
        const uint32_t* q = reinterpret_cast<const uint32_t*>(&s.w.heap[c]);
        lo = q[0];  // key, low word
        hi = q[1];
        sq = q[2];  // seq
    }
    const uint32_t mh = wave_min_u32(valid ? hi : ~0u);
    const bool c1 = valid && hi == mh;
    const uint32_t ml = wave_min_u32(c1 ? lo : ~0u);
    const bool c2 = c1 && lo == ml;
    const uint32_t ms = wave_min_u32(c2 ? sq : ~0u);
    const uint64_t m = ballot(c2 && sq == ms);  // seq is unique: one lane
    return first + (uint32_t)__builtin_ctzll(m);
}
__device__ __forceinline__ void heap_push(Sweep& s, const Ev& e) {
    if (s.heap_n >= s.w.heap_cap &&
        !migrate(s, s.w.heap, s.w.heap_cap, s.w.heap_g, s.w.heap_gcap, s.heap_n)) {
        fail(s, ST_RETRY);
        return;
    }
    Heap h;
    h.key = pkey(e.pos);
    h.seq = s.heap_seq++;
    h._pad = 0;
    h.ev = e;
    uint32_t i = s.heap_n++;
    gsync(s);
    while (i > 0) {
        uint32_t p = (i - 1) >> 6;
        Heap hp = ld(&s.w.heap[p]);
        if (!heap_less(h, hp)) break;
        put_nf(s, s.w.heap, i, hp);  // slots written here are never read in this sift
        i = p;
    }
    put_nf(s, s.w.heap, i, h);
    gsync(s);
}
__device__ __forceinline__ Heap heap_pop(Sweep& s) {
    gsync(s);
    Heap top = ld(&s.w.heap[0]);
    s.heap_n -= 1;
    if (s.heap_n > 0) {
        Heap last = ld(&s.w.heap[s.heap_n]);
        uint32_t i = 0;
        for (;;) {
            const uint64_t first = 64ull * i + 1;
            if (first >= s.heap_n) break;
            const uint32_t c = heap_min_child(s, (uint32_t)first);
            Heap hc = ld(&s.w.heap[c]);
            if (!heap_less(hc, last)) break;
            put_nf(s, s.w.heap, i, hc);  // later levels only read the children of c > i
            i = c;
        }
        put_nf(s, s.w.heap, i, last);
        gsync(s);
    }
    return top;
}
// EventQueue::insert_sorted / insert_sibling / vertex_event_sorted (event_queue.rs:188-250):
// all of them only ever insert strictly after the current position.
__device__ __forceinline__ void insert_event(Sweep& s, vec2 pos, vec2 to, int32_t winding,
                                             bool is_edge) {
    Ev e{pos, to, winding, is_edge ? 1u : 0u};
    heap_push(s, e);
}

// ---- scan_active_edges (fill.rs:1045-1291) ----------------------------------------------
// Lane-parallel form of the "edges before the current point" loop: each lane classifies one
// active edge; the loop stops at the first non-merge edge that is not before the point.
__device__ uint32_t classify_before(const Sweep& s, const AE& e, bool* connecting) {
    // returns 1 = before, 0 = stop (connecting set if the stop is a connection)
    float cx = s.cp.x;
    *connecting = false;
    if (veq(s.cp, e.to)) {
        *connecting = true;
        return 0;
    }
    if (e.max_x() < cx) return 1;
    if (e.min_x() > cx) return 0;
    if (e.from.y == e.to.y) {
        *connecting = true;
        return 0;
    }
    float ex = e.solve_x_for_y(s.cp.y);
    if (ffabs(ex - cx) <= s.tol) {
        *connecting = true;
        return 0;
    }
    if (ex > cx) return 0;
    return 1;
}

// returns false on an InternalError (ordering)
__device__ __forceinline__ bool is_edge_connecting(Sweep& s, const AE& e, uint32_t idx, bool* conn) {
    if (veq(s.cp, e.to)) {
        *conn = true;
        return true;
    }
    float cx = s.cp.x;
    float mnx = e.min_x(), mxx = e.max_x();
    if (mxx + s.tol < cx || e.to.y < s.cp.y) return false;
    if (mnx > cx) {
        *conn = false;
        return true;
    }
    float ex;
    if (e.from.y != e.to.y) ex = e.solve_x_for_y(s.cp.y);
    else if (mxx >= cx && mnx <= cx) ex = cx;
    else ex = e.to.x;
    if (ffabs(ex - cx) <= s.tol) {
        if (s.n_split >= s.w.act_cap) {
            fail(s, ST_RETRY);
            *conn = false;
            return true;
        }
        put(s, s.w.to_split, s.n_split, idx);
        s.n_split += 1;
        *conn = true;
        return true;
    }
    if (ex < cx) return false;
    *conn = false;
    return true;
}

__device__ __forceinline__ void push_vev(Sweep& s, int32_t span, uint32_t side) {
    put(s, s.w.vev_span, s.n_vev, span);
    put(s, s.w.vev_side, s.n_vev, side);
    s.n_vev += 1;
}

__device__ __forceinline__ bool scan_active_edges(Sweep& s) {
    s.n_vev = s.n_split = s.n_end = 0;
    s.merge_event = s.split_event = s.merge_split_event = false;
    s.above_start = s.above_end = 0;
    s.wbp = wnew();
    const float cx = s.cp.x;
    bool connecting_edges = false;
    uint32_t idx = 0;
    WState winding = wnew();
    bool previous_was_merge = false;
    // Step 1, 64 edges at a time.
    bool stopped = false;
    for (uint32_t base = 0; base < s.n_act && !stopped; base += WAVE) {
        uint32_t i = base + s.lane;
        bool valid = i < s.n_act;
        AE e;
        uint32_t before = 0, merge = 0;
        bool conn = false;
        if (valid) {
            e = ld(&s.w.act[i]);
            merge = e.is_merge;
            if (!merge) before = classify_before(s, e, &conn);
        }
        uint64_t stopm = ballot(valid && !merge && !before);
        uint64_t validm = ballot(valid);
        int first_stop = stopm ? __builtin_ctzll(stopm) : 64;
        uint32_t nproc = first_stop < 64 ? (uint32_t)first_stop : (uint32_t)__builtin_popcountll(validm);
        // Winding over the processed prefix [base, base + nproc), as lyon's per-edge updates
        // (WindingState::update): a wave prefix sum of the windings (wrapping like i16), and
        // one span entered per edge after which the point is inside, plus one per merge.
        const uint64_t mergem = ballot(valid && merge);
        const bool take = valid && (uint32_t)s.lane < nproc;
        const uint32_t incl = incl_scan(take && !merge ? (uint32_t)e.winding : 0u);
        const int32_t number = (int16_t)(winding.number + (int32_t)incl);
        const bool in_l = take && !merge && rule_in(s.rule, number);
        winding.span_index += (int32_t)(__builtin_popcountll(ballot(in_l)) +
                                        __builtin_popcountll(ballot(take && merge)));
        if (nproc > 0) {
            const uint32_t last = nproc - 1;
            winding.number = (int16_t)(winding.number + (int32_t)readlane_u(incl, (int)last));
            winding.in = rule_in(s.rule, winding.number);
            previous_was_merge = ((mergem >> last) & 1ull) != 0;
        }
        idx = base + nproc;
        if (first_stop < 64) {
            stopped = true;
            connecting_edges = readlane_u(conn ? 1u : 0u, first_stop) != 0;
        }
    }
    s.above_start = idx;
    s.wbp = winding;
    if (previous_was_merge) {
        s.wbp.span_index -= 1;
        s.above_start -= 1;
        if (!connecting_edges) {
            push_vev(s, winding.span_index - 1, 1);
            push_vev(s, winding.span_index, 0);
            s.merge_split_event = true;
        }
    }
    s.split_event = !connecting_edges && winding.in && !s.merge_split_event;
    if (connecting_edges) {
        bool in_before = winding.in;
        bool first_connecting_edge = !previous_was_merge;
        for (uint32_t i = idx; i < s.n_act; ++i) {
            AE e = ld(&s.w.act[i]);
            if (e.is_merge) {
                if (!winding.in) return false;  // MergeVertexOutside
                put(s, s.w.to_end, s.n_end, winding.span_index);
                s.n_end += 1;
                winding.span_index += 1;
                idx += 1;
                first_connecting_edge = false;
                continue;
            }
            bool conn;
            if (!is_edge_connecting(s, e, idx, &conn)) return false;
            if (!conn) break;
            if (!first_connecting_edge && winding.in) {
                put(s, s.w.to_end, s.n_end, winding.span_index);
                s.n_end += 1;
            }
            wupdate(winding, s.rule, e.winding);
            if (winding.in && winding.span_index >= (int32_t)s.n_spans) return false;  // spans
            idx += 1;
            first_connecting_edge = false;
        }
        bool in_after = winding.in;
        if (in_before && in_after && s.n_below == 0 && s.n_split == 0) s.merge_event = true;
        if (in_before) push_vev(s, s.wbp.span_index, 1);
        if (in_after) push_vev(s, winding.span_index, 0);
    }
    s.above_end = idx;
    // check_remaining_edges (fill.rs:1295-1324), lane-parallel
    bool bad = false;
    for (uint32_t base = idx; base < s.n_act; base += WAVE) {
        uint32_t i = base + s.lane;
        bool b = false;
        if (i < s.n_act) {
            AE e = ld(&s.w.act[i]);
            if (!e.is_merge) {
                if (e.max_x() < cx) b = true;
                else if (veq(s.cp, e.to)) b = true;
                else if (e.min_x() < cx && e.solve_x_for_y(s.cp.y) < cx) b = true;
            }
        }
        if (ballot(b)) bad = true;
    }
    return !bad;
}

// ---- process_edges_above (fill.rs:1381-1452) ----------------------------------------------
__device__ __forceinline__ void process_edges_above(Sweep& s) {
    for (uint32_t k = 0; k < s.n_vev; ++k)
        span_vertex(s, s.w.vev_span[k], s.cp, s.cv, s.w.vev_side[k]);
    for (uint32_t k = 0; k < s.n_end; ++k) end_span(s, s.w.to_end[k], s.cp, s.cv);
    cleanup_spans(s);
    for (uint32_t k = 0; k < s.n_split; ++k) {
        uint32_t ei = s.w.to_split[k];
        AE e = ld(&s.w.act[ei]);
        if (s.n_below >= s.w.below_cap &&
            !migrate(s, s.w.below, s.w.below_cap, s.w.below_g, s.w.below_gcap, s.n_below)) {
            fail(s, ST_RETRY);
            return;
        }
        PE pe{e.to, slope(sub(e.to, s.cp)), e.winding};
        put(s, s.w.below, s.n_below, pe);
        s.n_below += 1;
        e.to = s.cp;
        put(s, s.w.act, ei, e);
    }
    if (s.merge_event) {
        AE e = ld(&s.w.act[s.above_start]);
        e.is_merge = 1;
        e.from = e.to;
        e.winding = 0;
        e.from_id = s.cv;
        put(s, s.w.act, s.above_start, e);
        s.above_start += 1;
    }
}

// ---- process_edges_below (fill.rs:1455-1524) ----------------------------------------------
// Stable insertion sort by slope (lyon sorts with sort_unstable_by; slopes that compare
// equal are then merged as coincident edges, so their relative order does not change the
// region).
__device__ __forceinline__ void sort_edges_below(Sweep& s) {
    for (uint32_t i = 1; i < s.n_below; ++i) {
        PE v = ld(&s.w.below[i]);
        uint32_t j = i;
        while (j > 0) {
            PE u = ld(&s.w.below[j - 1]);
            if (!(v.sort_key < u.sort_key)) break;
            put(s, s.w.below, j, u);
            --j;
        }
        put(s, s.w.below, j, v);
    }
}

// merge_coincident_edges (fill.rs:2046-2106)
__device__ __forceinline__ void merge_coincident_edges(Sweep& s, uint32_t a_idx, uint32_t b_idx) {
    PE a = s.w.below[a_idx], b = ld(&s.w.below[b_idx]);
    uint32_t lower, upper;
    bool split;
    int c = cmp_pos(a.to, b.to);
    if (c > 0) {
        lower = a_idx;
        upper = b_idx;
        split = true;
    } else if (c < 0) {
        lower = b_idx;
        upper = a_idx;
        split = true;
    } else {
        lower = a_idx;
        upper = b_idx;
        split = false;
    }
    PE up = ld(&s.w.below[upper]);
    PE lo = ld(&s.w.below[lower]);
    up.winding = (int16_t)(up.winding + lo.winding);
    put(s, s.w.below, upper, up);
    vec2 split_point = up.to;
    shift_left(s, s.w.below, lower, s.n_below, 1);
    s.n_below -= 1;
    if (!split) return;
    insert_event(s, split_point, lo.to, lo.winding, true);
}

// handle_coincident_edges_below (fill.rs:2016-2043)
__device__ __forceinline__ void handle_coincident_edges_below(Sweep& s) {
    if (s.n_below < 2) return;
    for (uint32_t k = s.n_below - 1; k-- > 0;) {
        if (k + 1 >= s.n_below) continue;
        float a = s.w.below[k].sort_key, b = s.w.below[k + 1].sort_key;
        bool close;
        if (ffabs(a) <= 1.0f) close = ffabs(a - b) < 0.00005f;
        else close = ffabs(1.0f / a - 1.0f / b) < 0.00005f;
        if (close) merge_coincident_edges(s, k, k + 1);
    }
}

// split_event (fill.rs:1563-1608)
__device__ __forceinline__ void split_event(Sweep& s, uint32_t left_idx, int32_t left_span) {
    AE l = s.w.act[left_idx], r = ld(&s.w.act[left_idx + 1]);
    int32_t right_span = left_span + 1;
    if (is_after(l.from, r.from)) begin_span(s, left_span, l.from, l.from_id);
    else begin_span(s, right_span, r.from, r.from_id);
    span_vertex(s, left_span, s.cp, s.cv, 1);
    span_vertex(s, right_span, s.cp, s.cv, 0);
}

__device__ __forceinline__ void process_edges_below(Sweep& s) {
    WState w = s.wbp;
    sort_edges_below(s);
    handle_coincident_edges_below(s);
    if (s.split_event) {
        if (s.above_start == 0 || s.above_start >= s.n_act) {
            fail(s, ST_INTERNAL);
            return;
        }
        split_event(s, s.above_start - 1, w.span_index);
    }
    bool first = true;
    for (uint32_t k = 0; k < s.n_below; ++k) {
        if (!first && w.in) begin_span(s, w.span_index, s.cp, s.cv);
        wupdate(w, s.rule, s.w.below[k].winding);
        first = false;
    }
}

// nextafter(y, +inf) for finite y.
__device__ __forceinline__ float next_up(float y) {
    uint32_t b = __builtin_bit_cast(uint32_t, y);
    if ((b & 0x7fffffffu) == 0) return __builtin_bit_cast(float, 1u);
    return __builtin_bit_cast(float, (b & 0x80000000u) ? b - 1u : b + 1u);
}

// ---- intersections (fill.rs:1611-1846) ---------------------------------------------------
// LineSegment<f64>::intersection_t (line.rs:217-252)
__device__ __forceinline__ bool isect_t(double afx, double afy, double atx, double aty,
                                        double bfx, double bfy, double btx, double bty,
                                        double* ta, double* tb) {
    if ((atx == btx && aty == bty) || (afx == bfx && afy == bfy) ||
        (afx == btx && afy == bty) || (atx == bfx && aty == bfy))
        return false;
    double v1x = atx - afx, v1y = aty - afy;
    double v2x = btx - bfx, v2y = bty - bfy;
    double c = v1x * v2y - v1y * v2x;
    if (c == 0.0) return false;
    double sign = c > 0.0 ? 1.0 : -1.0;
    double abs_c = fabs(c);
    double v3x = bfx - afx, v3y = bfy - afy;
    double t = (v3x * v2y - v3y * v2x) * sign;
    double u = (v3x * v1y - v3y * v1x) * sign;
    if (t < 0.0 || t > abs_c || u < 0.0 || u > abs_c) return false;
    *ta = t / abs_c;
    *tb = u / abs_c;
    return true;
}

__device__ __forceinline__ void process_intersection(Sweep& s, double ta, double tb, uint32_t ai, PE& eb) {
    double bfx = s.cp.x, bfy = s.cp.y, btx = eb.to.x, bty = eb.to.y;
    double one_t = 1.0 - tb;
    vec2 ip = mk((float)(one_t * bfx + tb * btx), (float)(one_t * bfy + tb * bty));
    AE ae = ld(&s.w.act[ai]);
    if (veq(s.cp, ip)) {
        ae.from = ip;
        put(s, s.w.act, ai, ae);
        return;
    }
    if (!is_after(ip, s.cp)) ip.y = next_up(s.cp.y);
    if (is_near(ip, eb.to)) ip = eb.to;
    else if (is_near(ip, ae.to)) ip = ae.to;
    bool flipped_active = false;
    if (!veq(ae.to, ip) && !veq(ae.from, ip)) {
        if (is_after(ae.to, ip)) {
            insert_event(s, ip, ae.to, ae.winding, true);
        } else {
            flipped_active = true;
            insert_event(s, ae.to, ip, -ae.winding, true);
        }
        ae.to = ip;
        put(s, s.w.act, ai, ae);
    }
    if (!veq(eb.to, ip) && !veq(s.cp, ip)) {
        if (is_after(eb.to, ip)) {
            insert_event(s, ip, eb.to, eb.winding, true);
        } else {
            insert_event(s, eb.to, ip, -eb.winding, true);
            if (flipped_active) insert_event(s, ip, mk(0.0f, 0.0f), 0, false);
        }
        eb.to = ip;
    }
}

__device__ __forceinline__ void handle_intersections(Sweep& s) {
    const uint32_t skip_a = s.above_start, skip_b = s.above_end;
    for (uint32_t k = 0; k < s.n_below; ++k) {
        PE e = ld(&s.w.below[k]);
        float bmin = ffmin(s.cp.x, e.to.x);
        float bmax = fmax_(s.cp.x, e.to.x);
        double bfx = s.cp.x, bfy = s.cp.y, btx = e.to.x, bty = e.to.y;
        // Lane-parallel search for the smallest tb; ties keep the lowest index (the
        // reference's strict `tb < tb_min` in index order).  Each lane keeps the best of
        // its own edges (i = lane, lane + 64, ...: a strict < keeps its lowest index),
        // then one wave minimum over (tb, index) picks the winner.
        double tb_l = 1.0, ta_l = 0.0;
        uint32_t i_l = NONE;
        for (uint32_t base = 0; base < s.n_act; base += WAVE) {
            uint32_t i = base + s.lane;
            if (i < s.n_act && !(i >= skip_a && i < skip_b)) {
                AE ae = ld(&s.w.act[i]);
                if (!ae.is_merge && !(bmin > ae.max_x()) && !(bmax < ae.min_x())) {
                    double ta, tb;
                    if (isect_t(ae.from.x, ae.from.y, ae.to.x, ae.to.y, bfx, bfy, btx, bty, &ta,
                                &tb)) {
                        if (tb > 0.0 && ta > 0.0 && ta <= 1.0 && tb < tb_l) {
                            tb_l = tb;
                            ta_l = ta;
                            i_l = i;
                        }
                    }
                }
            }
        }
        // tb is in (0, 1): as a positive double its bits order like its value
        const uint64_t tbits = i_l == NONE ? ~0ull : (uint64_t)__builtin_bit_cast(int64_t, tb_l);
        const uint32_t mh = wave_min_u32((uint32_t)(tbits >> 32));
        const bool c1 = (uint32_t)(tbits >> 32) == mh;
        const uint32_t ml = wave_min_u32(c1 ? (uint32_t)tbits : ~0u);
        const bool c2 = c1 && (uint32_t)tbits == ml;
        const uint32_t mi = wave_min_u32(c2 ? i_l : NONE);
        uint32_t best_i = NONE;
        double best_tb = 1.0, best_ta = 0.0;
        if (mi != NONE) {
            const int src = __builtin_ctzll(ballot(c2 && i_l == mi));
            best_i = mi;
            best_tb = __shfl(tb_l, src, WAVE);
            best_ta = __shfl(ta_l, src, WAVE);
        }
        if (best_i != NONE) {
            process_intersection(s, best_ta, best_tb, best_i, e);
            put(s, s.w.below, k, e);
        }
    }
}

// ---- update_active_edges (fill.rs:1527-1561) -----------------------------------------------
__device__ __forceinline__ void update_active_edges(Sweep& s) {
    if (!s.no_isect) handle_intersections(s);
    const uint32_t a = s.above_start, b = s.above_end;
    const uint32_t removed = b - a, added = s.n_below;
    const uint32_t n_new = s.n_act - removed + added;
    if (n_new > s.w.act_cap) {
        if (n_new > s.w.act_gcap ||
            !migrate(s, s.w.act, s.w.act_cap, s.w.act_g, s.w.act_gcap, s.n_act)) {
            fail(s, ST_RETRY);
            return;
        }
        // the scan lists are dead here; they follow the active edges' capacity
        s.w.to_split = s.w.to_split_g;
        s.w.to_end = s.w.to_end_g;
    }
    if (added > removed) shift_right(s, s.w.act, b, s.n_act, added - removed);
    else if (removed > added) shift_left(s, s.w.act, a + added, s.n_act, removed - added);
    for (uint32_t base = 0; base < added; base += WAVE) {
        uint32_t k = base + s.lane;
        if (k < added) {
            PE pe = ld(&s.w.below[k]);
            AE e;
            e.from = s.cp;
            e.to = pe.to;
            e.winding = pe.winding;
            e.is_merge = 0;
            e.from_id = s.cv;
            e._pad = 0;
            st(&s.w.act[a + k], e);
        }
        gsync(s);
    }
    s.n_act = n_new;
    s.n_below = 0;
}

// ---- recovery (fill.rs:1848-2007) -----------------------------------------------------------
__device__ __forceinline__ void sort_active_edges(Sweep& s) {
    // keys (x at the sweep line, edge index); insertion sort into act2 then copy back.
    float y = s.cp.y;
    float prev_x = __builtin_nanf("");
    bool has_merge = false;
    for (uint32_t i = 0; i < s.n_act; ++i) {
        AE e = ld(&s.w.act[i]);
        float key;
        if (e.is_merge) {
            has_merge = true;
            key = prev_x;
        } else {
            bool eq_to = e.to.y == y, eq_from = e.from.y == y;
            float x;
            if (eq_to && eq_from) x = (e.max_x() >= s.cp.x && e.min_x() <= s.cp.x) ? s.cp.x : e.min_x();
            else if (eq_from) x = e.from.x;
            else if (eq_to) x = e.to.x;
            else x = e.solve_x_for_y(y);
            key = fmax_(x, e.min_x());
            prev_x = x;
        }
        // lyon sorts with partial_cmp(..).unwrap(): a NaN key (a merge vertex ahead of
        // every edge) is a panic there, an InternalError here (fill.rs:1894)
        if (key != key && s.n_act >= 2) {
            fail(s, ST_INTERNAL);
            return;
        }
        // stable insertion of (key, e) into act2[0..i)
        uint32_t j = i;
        while (j > 0) {
            AE u = ld(&s.w.act2[j - 1]);
            float uk = __builtin_bit_cast(float, u._pad);
            bool before;  // should e go before u?
            if (key < uk) before = true;
            else if (key > uk || key != key || uk != uk) before = false;
            else if (!e.is_merge && !u.is_merge) {
                float se = slope(sub(e.to, e.from)), su = slope(sub(u.to, u.from));
                before = se > su;
            } else {
                before = !e.is_merge && u.is_merge;
            }
            if (!before) break;
            put(s, s.w.act2, j, u);
            --j;
        }
        AE ek = e;
        ek._pad = __builtin_bit_cast(uint32_t, key);
        put(s, s.w.act2, j, ek);
    }
    for (uint32_t i = 0; i < s.n_act; ++i) {
        AE e = ld(&s.w.act2[i]);
        e._pad = 0;
        put(s, s.w.act, i, e);
    }
    if (!has_merge) return;
    int32_t wn = 0;
    for (uint32_t i = 0; i < s.n_act; ++i) {
        AE e = ld(&s.w.act[i]);
        bool needs_swap;
        if (e.is_merge) {
            needs_swap = !rule_in(s.rule, wn);
        } else {
            wn = (int16_t)(wn + e.winding);
            needs_swap = false;
        }
        if (needs_swap) {
            int32_t w = wn;
            uint32_t k = i;
            while (k > 0) {
                AE a = ld(&s.w.act[k - 1]);
                w = (int16_t)(w - a.winding);
                AE b = ld(&s.w.act[k]);
                put(s, s.w.act, k, a);
                put(s, s.w.act, k - 1, b);
                if (rule_in(s.rule, w)) break;
                k -= 1;
            }
        }
    }
}

// sort_active_edges above, and recover_from_error's swap of a last merge edge, by one lane
// over arrays in memory; false where it is an InternalError.
__device__ __noinline__ bool sort_edges_serial(AE* act, AE* act2, uint32_t n, vec2 cp,
                                               uint32_t rule) {
    const float y = cp.y;
    float prev_x = __builtin_nanf("");
    bool has_merge = false;
    for (uint32_t i = 0; i < n; ++i) {
        AE e = ld(&act[i]);
        float key;
        if (e.is_merge) {
            has_merge = true;
            key = prev_x;
        } else {
            const bool eq_to = e.to.y == y, eq_from = e.from.y == y;
            float x;
            if (eq_to && eq_from) x = (e.max_x() >= cp.x && e.min_x() <= cp.x) ? cp.x : e.min_x();
            else if (eq_from) x = e.from.x;
            else if (eq_to) x = e.to.x;
            else x = e.solve_x_for_y(y);
            key = fmax_(x, e.min_x());
            prev_x = x;
        }
        if (key != key && n >= 2) return false;
        uint32_t j = i;
        while (j > 0) {
            const AE u = ld(&act2[j - 1]);
            const float uk = __builtin_bit_cast(float, u._pad);
            bool before;
            if (key < uk) before = true;
            else if (key > uk || key != key || uk != uk) before = false;
            else if (!e.is_merge && !u.is_merge)
                before = slope(sub(e.to, e.from)) > slope(sub(u.to, u.from));
            else before = !e.is_merge && u.is_merge;
            if (!before) break;
            st(&act2[j], u);
            --j;
        }
        e._pad = __builtin_bit_cast(uint32_t, key);
        st(&act2[j], e);
    }
    for (uint32_t i = 0; i < n; ++i) {
        AE e = ld(&act2[i]);
        e._pad = 0;
        st(&act[i], e);
    }
    if (has_merge) {
        int32_t wn = 0;
        for (uint32_t i = 0; i < n; ++i) {
            const AE e = ld(&act[i]);
            bool needs_swap = false;
            if (e.is_merge) needs_swap = !rule_in(rule, wn);
            else wn = (int16_t)(wn + e.winding);
            if (!needs_swap) continue;
            int32_t w = wn;
            for (uint32_t k = i; k > 0; --k) {
                const AE a = ld(&act[k - 1]), b = ld(&act[k]);
                w = (int16_t)(w - a.winding);
                st(&act[k], a);
                st(&act[k - 1], b);
                if (rule_in(rule, w)) break;
            }
        }
    }
    if (n > 1 && act[n - 1].is_merge) {
        const AE a = ld(&act[n - 1]), b = ld(&act[n - 2]);
        st(&act[n - 1], b);
        st(&act[n - 2], a);
    }
    return true;
}

__device__ __forceinline__ void recover_from_error(Sweep& s) {
    sort_active_edges(s);
    uint32_t len = s.n_act;
    if (len > 1 && s.w.act[len - 1].is_merge) {
        AE a = s.w.act[len - 1], b = ld(&s.w.act[len - 2]);
        put(s, s.w.act, len - 1, b);
        put(s, s.w.act, len - 2, a);
    }
    WState w = wnew();
    for (uint32_t i = 0; i < s.n_act; ++i) {
        AE e = ld(&s.w.act[i]);
        if (e.is_merge) w.span_index += 1;
        else wupdate(w, s.rule, e.winding);
        if (w.span_index >= (int32_t)s.n_spans) begin_span(s, w.span_index, e.from, e.from_id);
    }
    while ((int64_t)s.n_spans > (int64_t)w.span_index + 1) s.n_spans -= 1;
}

__device__ __forceinline__ bool process_events(Sweep& s) {
    if (!scan_active_edges(s)) return false;
    process_edges_above(s);
    process_edges_below(s);
    update_active_edges(s);
    return true;
}

// ---- event generation: EventQueueBuilder (event_queue.rs:451-905) ---------------------------
struct Builder {
    vec2 current, prev, second;
    uint32_t nth;
    uint32_t n;  // events written
};

__device__ __forceinline__ void b_push(Sweep& s, Builder& b, vec2 pos, vec2 to, int32_t w,
                                       bool is_edge) {
    if (b.n < s.w.ev_cap) {
        if (s.lane == 0) {
            st(&s.w.ev[b.n], Ev{pos, to, w, is_edge ? 1u : 0u});
            s.w.key_a[b.n] = pkey(pos);
            s.w.idx_a[b.n] = b.n;
        }
    } else {
        fail(s, ST_RETRY);
    }
    b.n++;
}
__device__ __forceinline__ void b_vertex(Sweep& s, Builder& b, vec2 at) {
    b_push(s, b, at, mk(__builtin_nanf(""), __builtin_nanf("")), 0, false);
}
// add_edge (:693-726)
__device__ __forceinline__ void b_edge(Sweep& s, Builder& b, vec2 from, vec2 to, int32_t w) {
    if (veq(from, to)) return;
    vec2 pos = from, dst = to;
    if (is_after(pos, to)) {
        dst = pos;
        pos = to;
        w = -w;
    }
    b_push(s, b, pos, dst, w, true);
    b.nth += 1;
}
// line_segment (:728-756)
__device__ __forceinline__ void b_line(Sweep& s, Builder& b, vec2 to) {
    vec2 from = b.current;
    if (veq(from, to)) return;
    if (is_after(from, to) && b.nth > 0 && is_after(from, b.prev)) b_vertex(s, b, from);
    if (b.nth == 0) b.second = to;
    b_edge(s, b, from, to, 1);
    b.prev = b.current;
    b.current = to;
}
// quadratic_bezier_segment / cubic_bezier_segment (:758-900): flatten the curve oriented
// downwards; emit edges and the vertex events found between them.
__device__ __forceinline__ void b_curve(Sweep& s, Builder& b, bool cubic, vec2 c1, vec2 c2, vec2 to, float tol) {
    vec2 ofrom = b.current;
    bool needs_swap = is_after(ofrom, to);
    vec2 f = ofrom, a = c1, bb = c2, t = to;
    if (needs_swap) {
        vec2 x = f;
        f = t;
        t = x;
        if (cubic) {
            x = a;
            a = bb;
            bb = x;
        }
    }
    int32_t winding = needs_swap ? -1 : 1;
    vec2 prev = f;
    bool have_first = false;
    vec2 first = mk(0.0f, 0.0f);
    bool is_first_edge = b.nth == 0;
    // polynomial form and Wang count (quadratic_bezier.rs:891-974, cubic_bezier.rs:1318-1403)
    float n = cubic ? cubic_wang(f, a, bb, t, tol) : quad_wang(f, a, t, tol);
    float step = 1.0f / n;
    uint32_t cnt = seg_count(n);
    vec2 a0 = f, a1, a2, a3 = mk(0.0f, 0.0f);
    if (cubic) {
        a1 = mul(sub(a, f), 3.0f);
        a2 = add(sub(mul(f, 3.0f), mul(a, 6.0f)), mul(bb, 3.0f));
        a3 = add(sub(t, f), mul(sub(a, bb), 3.0f));
    } else {
        a1 = mul(sub(a, f), 2.0f);
        a2 = sub(add(f, t), mul(a, 2.0f));
    }
    float t0 = 0.0f;
    vec2 lf = f;
    for (uint32_t i = 0; i < cnt && s.status == ST_OK; ++i) {
        vec2 lt;
        if (i + 1 == cnt) {
            lt = t;
        } else {
            float t1 = t0 + step;
            vec2 v = a0;
            float tt = t1;
            v = add(v, mul(a1, tt));
            tt = tt * t1;
            v = add(v, mul(a2, tt));
            if (cubic) {
                tt = tt * t1;
                v = add(v, mul(a3, tt));
            }
            lt = v;
            t0 = t1;
        }
        if (!veq(lf, lt)) {
            if (!have_first) {
                have_first = true;
                first = lt;
            } else if (is_after(lf, lt) && is_after(lf, prev)) {
                b_vertex(s, b, lf);
            }
            b_edge(s, b, lf, lt, winding);
            prev = lf;
        }
        lf = lt;
    }
    if (have_first) {
        vec2 second = needs_swap ? prev : first;
        vec2 previous = needs_swap ? first : prev;
        if (is_first_edge) b.second = second;
        else if (is_after(ofrom, b.prev) && is_after(ofrom, second)) b_vertex(s, b, ofrom);
        b.prev = previous;
        b.current = to;
    }
}
// end (:661-682)
__device__ __forceinline__ void b_end(Sweep& s, Builder& b, vec2 first) {
    if (b.nth == 0) return;
    b_line(s, b, first);
    if (is_after(first, b.prev) && is_after(first, b.second)) b_vertex(s, b, first);
    b.nth = 0;
}

// ---- stable LSD radix sort of (key, idx), 8 bits per pass ---------------------------------
__device__ __forceinline__ void radix_sort(Sweep& s, uint32_t n, uint32_t* hist /* LDS, 256 */) {
    uint64_t* ksrc = s.w.key_a;
    uint32_t* isrc = s.w.idx_a;
    uint64_t* kdst = s.w.key_b;
    uint32_t* idst = s.w.idx_b;
    for (int pass = 0; pass < 8; ++pass) {
        const int shift = pass * 8;
        for (int d = s.lane; d < 256; d += WAVE) hist[d] = 0;
        gsync(s);
        // counts per digit: the lanes of a chunk with equal digits (peers, from one ballot
        // per digit bit) add their number once, through their lowest lane, so the updates
        // of a chunk go to distinct counters (no atomics, no serialised equal addresses)
        for (uint32_t base = 0; base < n; base += WAVE) {
            const uint32_t i = base + s.lane;
            const bool valid = i < n;
            const uint32_t d = valid ? (uint32_t)(ksrc[i] >> shift) & 255u : 0u;
            uint64_t peers = ballot(valid);
            for (int bit = 0; bit < 8; ++bit) {
                const uint64_t m = ballot(valid && ((d >> bit) & 1u));
                peers &= ((d >> bit) & 1u) ? m : ~m;
            }
            if (valid && (uint32_t)__builtin_ctzll(peers) == (uint32_t)s.lane)
                hist[d] += (uint32_t)__builtin_popcountll(peers);
            gsync(s);
        }
        // exclusive scan of 256 counters (4 per lane)
        uint32_t c[4], tot = 0;
        for (int q = 0; q < 4; ++q) {
            c[q] = hist[4 * s.lane + q];
            tot += c[q];
        }
        uint32_t incl = incl_scan(tot);
        uint32_t run = incl - tot;
        gsync(s);
        for (int q = 0; q < 4; ++q) {
            hist[4 * s.lane + q] = run;
            run += c[q];
        }
        gsync(s);
        // stable scatter: rank among equal digits within the 64-element chunk
        for (uint32_t base = 0; base < n; base += WAVE) {
            uint32_t i = base + s.lane;
            bool valid = i < n;
            uint64_t k = valid ? ksrc[i] : 0;
            uint32_t d = (uint32_t)(k >> shift) & 255u;
            uint64_t peers = ballot(valid);
            for (int bit = 0; bit < 8; ++bit) {
                uint64_t m = ballot(valid && ((d >> bit) & 1u));
                peers &= ((d >> bit) & 1u) ? m : ~m;
            }
            uint32_t rank = __builtin_popcountll(peers & mask_lt(s.lane));
            uint32_t basepos = valid ? hist[d] : 0;
            gsync(s);
            if (valid) {
                kdst[basepos + rank] = k;
                idst[basepos + rank] = isrc[i];
            }
            // the highest lane of every peer group advances the digit's offset
            bool leader = valid && (highest_bit(peers) == s.lane);
            if (leader) hist[d] = basepos + (uint32_t)__builtin_popcountll(peers);
            gsync(s);
        }
        uint64_t* tk = ksrc;
        ksrc = kdst;
        kdst = tk;
        uint32_t* ti = isrc;
        isrc = idst;
        idst = ti;
    }
    // 8 passes: the sorted data ends in key_a/idx_a again.
}

// The path's events in sweep order (set_path, event_queue.rs:483-551): s.w.ev, with the
// sorted keys in s.w.key_a and the events' indices in s.w.idx_a; s.n_static.
__device__ __forceinline__ uint32_t make_events(Sweep& s, const PathBatchDev& in, uint32_t path,
                                                const lyg_fill_options& o, uint32_t* hist) {
    const uint32_t vb = in.verb_off[path], ve = in.verb_off[path + 1];
    const uint32_t pb = in.point_off[path], pe = in.point_off[path + 1];
    const uint8_t* verbs = in.verbs + vb;
    const float2* pts = reinterpret_cast<const float2*>(in.points) + pb;
    const uint32_t npts = pe - pb;
    const bool horiz = o.sweep_orientation == LYG_ORIENT_HORIZONTAL;
    auto pt = [&](uint32_t i) -> vec2 {
        if (i >= npts) return mk(__builtin_nanf(""), __builtin_nanf(""));
        float2 q = pts[i];
        vec2 p = mk(q.x, q.y);
        return horiz ? mk(-p.y, p.x) : p;  // event_queue.rs:12-15
    };
    // ---- events (set_path, event_queue.rs:483-551) ----
    Builder b;
    b.current = b.prev = b.second = mk(__builtin_nanf(""), __builtin_nanf(""));
    b.nth = 0;
    b.n = 0;
    uint32_t p = 0;
    vec2 first = mk(0.0f, 0.0f);
    for (uint32_t v = 0; v < ve - vb && s.status == ST_OK; ++v) {
        uint8_t verb = verbs[v];
        if (verb == LYG_VERB_BEGIN) {
            vec2 at = pt(p++);
            first = at;
            b.nth = 0;
            b.current = at;
        } else if (verb == LYG_VERB_LINE) {
            b_line(s, b, pt(p++));
        } else if (verb == LYG_VERB_QUADRATIC) {
            vec2 c = pt(p), t = pt(p + 1);
            p += 2;
            b_curve(s, b, false, c, c, t, o.tolerance);
        } else if (verb == LYG_VERB_CUBIC) {
            vec2 c1 = pt(p), c2 = pt(p + 1), t = pt(p + 2);
            p += 3;
            b_curve(s, b, true, c1, c2, t, o.tolerance);
        } else {
            if (verb == LYG_VERB_CLOSE) p++;
            b_end(s, b, first);
        }
    }
    gsync(s);
    if (s.status != ST_OK) return s.status;
    s.n_static = b.n;
    // NaN positions end the tessellation with PositionIsNaN (fill.rs:884-888).
    {
        bool nanb = false;
        for (uint32_t base = 0; base < s.n_static; base += WAVE) {
            uint32_t i = base + s.lane;
            bool bad = false;
            if (i < s.n_static) {
                Ev e = ld(&s.w.ev[i]);
                bad = (e.pos.x != e.pos.x) || (e.pos.y != e.pos.y);
            }
            if (ballot(bad)) nanb = true;
        }
        if (nanb) return ST_POSITION_NAN;
    }
    radix_sort(s, s.n_static, hist);
    return ST_OK;
}

}  // namespace fillk

}  // namespace lyg
