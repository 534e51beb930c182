// Host side of the variable-width stroke (StrokeOptions::variable_line_width): the plan and
// its scans, the count, the offset scans, the output check, the emit launches; the serial
// kernel (one lane per path) for the paths the parallel form leaves out.
#include <algorithm>
#include <vector>

#include "ctx.h"
#include "internal.h"
#include "lyg_types.h"

extern "C" {
hipError_t lyg_launch_stroke_vw(const lyg::StrokeVWLaunch* L, int emit, int grid,
                                hipStream_t s);
hipError_t lyg_launch_vw_plan(const lyg::VWPar* P, int grid, hipStream_t s);
hipError_t lyg_launch_vw_count(const lyg::VWPar* P, int grid_paths, int grid_win, uint32_t chunk,
                               hipStream_t s);
hipError_t lyg_launch_vw_totals(const lyg::VWPar* P, hipStream_t s);
hipError_t lyg_launch_vw_emit(const lyg::VWPar* P, int grid_win, uint32_t chunk, hipStream_t s);
hipError_t lyg_launch_fill_u32(uint32_t* p, uint32_t n, uint32_t v, hipStream_t s);
hipError_t lyg_launch_scan_several(const lyg::ScanJobs* J, hipStream_t s);
}

namespace {

bool valid_opts(const lyg_stroke_options& o) {
    return o.start_cap <= 2 && o.end_cap <= 2 && o.line_join <= 3;
}

// Scans of up to 32,768 counts each in one launch, a block each; longer ones one by one.
bool scans(lyg_ctx* c, std::initializer_list<lyg::ScanJob> jobs, uint32_t* overflow) {
    lyg::ScanJobs J{};
    J.overflow = overflow;
    bool small = true;
    for (const lyg::ScanJob& j : jobs) {
        J.job[J.n_jobs++] = j;
        small = small && j.n <= 32768;
    }
    if (small) return check(c, lyg_launch_scan_several(&J, c->stream), "scans");
    for (const lyg::ScanJob& j : jobs)
        if (!check(c, ctx_scan(c, j.counts, j.n, j.offsets, j.total, overflow, c->stream), "scan"))
            return false;
    return true;
}

// Launch shape of the window kernels.
struct VWShape {
    int grid_paths, grid;
    uint32_t chunk;  // consecutive windows per wave and turn
};

// Points of a batch beyond which it goes to the serial kernel (the parallel form keeps 17
// bytes per flattened point, the output takes about 40).
constexpr uint64_t VW_MAX_POINTS = 1ull << 30;

// Paths of no more points are sooner walked by a lane each (13 us a point) than by the parallel
// form's launches, while every path has a wave: plain calls of 1 / 3 / 10 lines 168 187 279 us
// against 220 to 250.
constexpr uint32_t VW_FEW = 5;

// About six resident waves per SIMD (four SIMDs per CU) of the serial kernel.
uint32_t serial_slots(const lyg_ctx* c) { return (uint32_t)std::max(1, c->cu_count) * 4u * 6u; }

// The plan and the parallel form's memory.  LYG_ERR_NO_SPACE: the batch goes to the serial
// kernel (too many points, or no device memory for them; no path for the parallel form; few
// short paths).
int32_t vw_plan(lyg_ctx* c, const lyg::StrokeVWLaunch& L, uint32_t n, bool want_attrs,
                lyg::VWPar* out, VWShape* sh) {
    hipStream_t s = c->stream;
    lyg::VWPar P{};
    P.in = L.in;
    P.opts = L.opts;
    P.opts_stride = L.opts_stride;
    P.widths = L.widths;
    P.widths_stride = L.widths_stride;
    P.attrs = L.attrs;
    P.n_attrs = L.n_attrs;
    P.path_status = L.path_status;
    P.path_nv = L.path_nv;
    P.path_ni = L.path_ni;
    P.err = L.err;
    if (!ensure(c, c->vw_path, 4ull * (11ull * n + 4) + 64)) {
        (void)hipGetLastError();
        return LYG_ERR_NO_SPACE;
    }
    uint32_t* u = as<uint32_t>(c->vw_path);
    auto take = [&](size_t k) {
        uint32_t* p = u;
        u += k;
        return p;
    };
    P.few = VW_FEW;
    P.ctr = take(16);
    P.raw_n = take(n);
    P.win_n = take(n);
    P.tail_n = take(n);
    P.att_cap_n = take(n);
    P.kept_n = take(n);
    P.path_mode = take(n);
    P.slow_list = take(n);
    uint32_t* off[4];
    for (uint32_t*& o : off) o = take((size_t)n + 1);
    P.raw_off = off[0];
    P.win_off = off[1];
    P.tail_off = off[2];
    P.att_off = off[3];
    sh->grid_paths = (int)std::min<uint32_t>(n, (uint32_t)std::max(1, c->cu_count) * 32u);
    if (!check(c, lyg_launch_fill_u32(P.ctr, 16, 0, s), "reset") ||
        !check(c, lyg_launch_vw_plan(&P, sh->grid_paths, s), "stroke vw plan") ||
        !scans(c, {{P.raw_n, n, off[0], c->d_totals + 2}, {P.win_n, n, off[1], c->d_totals + 3},
                   {P.tail_n, n, off[2], c->d_totals + 4},
                   {P.att_cap_n, n, off[3], c->d_totals + 5}}, P.ctr + 8))
        return LYG_ERR_DEVICE;
    uint64_t* h = reinterpret_cast<uint64_t*>(c->h_pinned);
    h[4] = 1;
    if (!check(c, hipMemcpyAsync(h, c->d_totals + 2, 32, hipMemcpyDeviceToHost, s), "D2H") ||
        (n <= serial_slots(c) &&
         !check(c, hipMemcpyAsync(h + 4, P.ctr + 5, 4, hipMemcpyDeviceToHost, s), "D2H")) ||
        !check(c, hipStreamSynchronize(s), "sync"))
        return LYG_ERR_DEVICE;
    if (h[0] == 0 || (uint32_t)h[4] == 0) return LYG_ERR_NO_SPACE;
    const uint64_t raw = h[0], win = h[1], tails = h[2], att = h[3];
    if (raw > VW_MAX_POINTS || tails > VW_MAX_POINTS || att > VW_MAX_POINTS)
        return LYG_ERR_NO_SPACE;
    P.n_windows = (uint32_t)win;
    P.n_tails = (uint32_t)tails;
    // candidates for skipped joins: but for rounding, each is a curve's first point, and a curve
    // has an edge with side lines at both ends
    P.cand_cap = (uint32_t)std::max<uint64_t>({4096, win, att / 2});
    P.dirty_cap = 4u * P.cand_cap;
    const bool src = want_attrs;
    if (!ensure(c, c->vw_rec, 16 * raw) || !ensure(c, c->vw_flags, raw) ||
        (src && !ensure(c, c->vw_src, 12 * raw)) || !ensure(c, c->vw_att, 20 * att) ||
        !ensure(c, c->vw_win, 4 * (5 * win + 2)) ||
        !ensure(c, c->vw_tails, sizeof(lyg::VWTail) * tails) ||
        !ensure(c, c->vw_lists, 4ull * (2ull * P.cand_cap + P.dirty_cap))) {
        (void)hipGetLastError();  // the serial kernel needs none of it
        return LYG_ERR_NO_SPACE;
    }
    P.rec = as<float>(c->vw_rec);
    P.pflags = as<uint8_t>(c->vw_flags);
    if (src) {
        P.src_t = as<float>(c->vw_src);
        P.src_id = as<uint32_t>(c->vw_src) + raw;
    }
    P.att_n = as<float>(c->vw_att);
    P.att_point = as<uint32_t>(c->vw_att) + 4 * att;
    if (!check(c, lyg_launch_fill_u32(P.att_point, (uint32_t)att, 0xffffffffu, s), "reset"))
        return LYG_ERR_DEVICE;
    u = as<uint32_t>(c->vw_win);
    P.win_att = take(win);
    P.win_nv = take(win);
    P.win_ni = take(win);
    P.win_voff = take(win + 1);
    P.win_ioff = take(win + 1);
    P.tails = as<lyg::VWTail>(c->vw_tails);
    P.cands = as<uint32_t>(c->vw_lists);
    P.dirty = P.cands + 2ull * P.cand_cap;
    // windows: 8 resident blocks of four waves per CU, a few consecutive windows per wave and
    // turn (they share the search for their path)
    const uint32_t blocks = (uint32_t)std::max(1, c->cu_count) * 8u;
    sh->chunk = std::min<uint32_t>(16u, std::max<uint32_t>(1u, P.n_windows / (blocks * 16u)));
    const uint64_t turns = (win + 4ull * sh->chunk - 1) / (4ull * sh->chunk);
    sh->grid = (int)std::max<uint64_t>(1, std::min<uint64_t>(turns, blocks));
    *out = P;
    return LYG_OK;
}

// Counts of the planned batch into path_nv / path_ni (of the paths not left to the serial
// kernel).
int32_t vw_count(lyg_ctx* c, lyg::VWPar& P, const VWShape& sh) {
    hipStream_t s = c->stream;
    uint32_t* wv = const_cast<uint32_t*>(P.win_voff);
    uint32_t* wi = const_cast<uint32_t*>(P.win_ioff);
    if (!check(c, lyg_launch_vw_count(&P, sh.grid_paths, sh.grid, sh.chunk, s),
               "stroke vw count") ||
        !scans(c, {{P.win_nv, P.n_windows, wv, c->d_totals + 6},
                   {P.win_ni, P.n_windows, wi, c->d_totals + 7}}, P.ctr + 8) ||
        !check(c, lyg_launch_vw_totals(&P, s), "stroke vw totals"))
        return LYG_ERR_DEVICE;
    return LYG_OK;
}

// Runs the batch `L` (inputs, options, widths set), `serial`: without the plan; offsets go to vtx_off / idx_off (n + 1
// each), per-path statuses to c->f_status; want_attrs: vertex attributes will be asked for
// (L.out_attrs is set by then); `alloc` sets the output arrays once the totals
// are known.
int32_t stroke_vw_run(lyg_ctx* c, lyg::StrokeVWLaunch& L, bool serial, bool want_attrs,
                      uint32_t* vtx_off, uint32_t* idx_off, uint32_t vertex_offset, const lygi::OutAlloc& alloc,
                      uint64_t* tv, uint64_t* ti, std::vector<uint32_t>* status) {
    const uint32_t n = L.in.n_paths;
    hipStream_t s = c->stream;
    if (!ensure(c, c->counts_v, 4ull * n) || !ensure(c, c->counts_i, 4ull * n) ||
        !ensure(c, c->f_status, 4ull * n))
        return LYG_ERR_DEVICE;
    L.path_nv = as<uint32_t>(c->counts_v);
    L.path_ni = as<uint32_t>(c->counts_i);
    L.path_status = as<uint32_t>(c->f_status);
    L.vertex_offset = vertex_offset;
    L.err = c->d_counters + 5;
    lyg::VWPar P{};
    VWShape sh{};
    int32_t st = serial || c->vw_serial ? (int32_t)LYG_ERR_NO_SPACE
                                        : vw_plan(c, L, n, want_attrs, &P, &sh);
    if (st == LYG_OK) st = vw_count(c, P, sh);
    if (st == LYG_ERR_DEVICE) return st;
    bool par = st == LYG_OK;
    // the serial kernel, over all paths or those left to it: its waves take as few as fill them
    const uint32_t slots = serial_slots(c);
    int grid = 0;
    uint64_t* h = reinterpret_cast<uint64_t*>(c->h_pinned);
    status->assign(n, 0);
    for (;;) {
        L.list = par ? P.slow_list : nullptr;
        L.n_list = par ? P.ctr + 1 : nullptr;
        L.paths_per_wave =  // of a list: by its length, in the kernel
            std::min<uint32_t>(64u, std::max<uint32_t>(1u, (n + slots - 1) / slots));
        grid = par ? (int)std::min(n, slots)
                   : (int)std::min<uint32_t>((n + L.paths_per_wave - 1) / L.paths_per_wave,
                                             1u << 20);
        h[3] = h[4] = 0;  // serial paths, candidates, windows counted again, a list overflowed
        uint32_t* went = reinterpret_cast<uint32_t*>(h + 3);
        if (!check(c, lyg_launch_fill_u32(c->d_counters + 4, 2, 0, s), "reset") ||
            !check(c, lyg_launch_stroke_vw(&L, 0, grid, s), "stroke vw count") ||
            !scans(c, {{L.path_nv, n, vtx_off, c->d_totals + 0},
                       {L.path_ni, n, idx_off, c->d_totals + 1}}, c->d_counters + 4) ||
            !check(c, hipMemcpyAsync(h, c->d_totals, 16, hipMemcpyDeviceToHost, s), "D2H") ||
            !check(c, hipMemcpyAsync(h + 2, c->d_counters + 4, 4, hipMemcpyDeviceToHost, s),
                   "D2H") ||
            (par && !check(c, hipMemcpyAsync(went, P.ctr + 1, 16, hipMemcpyDeviceToHost, s),
                           "D2H")) ||
            !check(c, hipMemcpyAsync(status->data(), L.path_status, 4ull * n,
                                     hipMemcpyDeviceToHost, s),
                   "D2H") ||
            !check(c, hipStreamSynchronize(s), "sync"))
            return LYG_ERR_DEVICE;
        c->last_vw_serial = par && !went[3] ? went[0] : n;
        c->last_vw_recounted = went[2];
        if (!went[3]) break;
        par = false;  // more joins that may fold back than the lists hold
    }
    *tv = h[0];
    *ti = h[1];
    if ((uint32_t)h[2]) return LYG_ERR_TOO_MANY_VERTICES;
    // BuffersBuilder::add_vertex_impl: ids up to u32::MAX - 1 (geometry_builder.rs:338-350)
    if (*tv > 0 && (uint64_t)vertex_offset + *tv - 1 > 0xfffffffeull)
        return LYG_ERR_TOO_MANY_VERTICES;
    float* ov = nullptr;
    uint32_t* oi = nullptr;
    st = alloc(*tv, *ti, &ov, &oi);
    if (st != LYG_OK) return st;
    L.vtx_off = vtx_off;
    L.idx_off = idx_off;
    L.out_vertices = ov;
    L.out_indices = oi;
    if (par) {
        P.vtx_off = vtx_off;
        P.idx_off = idx_off;
        P.out_vertices = ov;
        P.out_indices = oi;
        P.out_attrs = L.out_attrs;
        P.vertex_offset = vertex_offset;
        if (!check(c, lyg_launch_vw_emit(&P, sh.grid, sh.chunk, s), "stroke vw emit"))
            return LYG_ERR_DEVICE;
    }
    uint32_t err = 0;
    if (!check(c, lyg_launch_stroke_vw(&L, 1, grid, s), "stroke vw emit") ||
        !check(c, hipMemcpyAsync(&err, c->d_counters + 5, 4, hipMemcpyDeviceToHost, s), "D2H") ||
        !check(c, hipStreamSynchronize(s), "sync"))
        return LYG_ERR_DEVICE;
    // the emit pass wrote past its path's counted range: the two passes disagreed
    if (err) return LYG_ERR_INTERNAL;
    return LYG_OK;
}

int32_t first_failure(const std::vector<uint32_t>& st) {
    for (uint32_t v : st)
        if (v) return (int32_t)v;
    return LYG_OK;
}

}  // namespace

extern "C" {

// Not in lyg.h: sends every path to the serial kernel (the two forms give the same bytes); how
// the last call went: paths walked by it, and windows counted again for joins that fold back.
void lyg_ctx_set_vw_serial(lyg_ctx* c, int enabled) { c->vw_serial = enabled != 0; }
void lyg_ctx_last_vw(const lyg_ctx* c, uint32_t* serial, uint32_t* recounted) {
    *serial = c->last_vw_serial;
    *recounted = c->last_vw_recounted;
}

// StrokeTessellator::tessellate_path with StrokeOptions::variable_line_width
// (stroke.rs:653-767) for a batch in device memory.
int32_t lyg_stroke_batch_vw(lyg_ctx* c, const lyg_batch_in* in, const float* attributes,
                            uint32_t n_attributes, uint32_t width_attribute,
                            const lyg_stroke_options* opts, uint32_t n_opts, lyg_batch_out* out,
                            float* out_attributes) {
    if (!c || !in || !opts || !out || !attributes) return LYG_ERR_INVALID_ARGUMENT;
    if (n_opts != 1 && n_opts != in->n_paths) return LYG_ERR_INVALID_ARGUMENT;
    if (width_attribute >= n_attributes) return LYG_ERR_INVALID_ARGUMENT;
    out->n_vertices = 0;
    out->n_indices = 0;
    if (in->n_paths == 0) return LYG_OK;
    if (!out->path_vertex_offsets || !out->path_index_offsets) return LYG_ERR_INVALID_ARGUMENT;
    if (!check(c, hipSetDevice(c->device), "hipSetDevice")) return LYG_ERR_DEVICE;
    lyg::StrokeVWLaunch L{};
    L.in.verbs = in->verbs;
    L.in.points = in->points;
    L.in.verb_off = in->verb_offsets;
    L.in.point_off = in->point_offsets;
    L.in.n_paths = in->n_paths;
    L.opts = opts;
    L.opts_stride = n_opts == 1 ? 0 : 1;
    L.widths = attributes + width_attribute;
    L.widths_stride = n_attributes;
    L.attrs = attributes;
    L.n_attrs = n_attributes;
    L.out_attrs = out_attributes;
    uint64_t tv = 0, ti = 0;
    std::vector<uint32_t> status;
    int32_t st = stroke_vw_run(
        c, L, false, out_attributes != nullptr, out->path_vertex_offsets, out->path_index_offsets,
        out->vertex_offset,
        [&](uint64_t nv, uint64_t ni, float** v, uint32_t** i) -> int32_t {
            if (nv > out->vertex_capacity || ni > out->index_capacity) return LYG_ERR_CAPACITY;
            *v = out->vertices;
            *i = out->indices;
            return LYG_OK;
        },
        &tv, &ti, &status);
    out->n_vertices = tv;
    out->n_indices = ti;
    if (out->path_status && !status.empty() &&
        !check(c, hipMemcpy(out->path_status, status.data(), 4ull * in->n_paths,
                            hipMemcpyHostToDevice),
               "H2D"))
        return LYG_ERR_DEVICE;
    if (st != LYG_OK) return st;
    return first_failure(status);
}

// The same for one path in host memory (tessellate_path into caller-owned arrays);
// attributes: n_points x n_attributes floats.
int32_t lyg_stroke_path_vw(lyg_ctx* c, const lyg_path_view* path, const float* attributes,
                           uint32_t n_attributes, uint32_t width_attribute,
                           const lyg_stroke_options* opts, lyg_output* out,
                           float* out_attributes) {
    if (!c || !path || !opts || !out) return LYG_ERR_INVALID_ARGUMENT;
    if (!valid_opts(*opts) || width_attribute >= n_attributes) return LYG_ERR_INVALID_ARGUMENT;
    if ((path->n_verbs && !path->verbs) || (path->n_points && !path->points) ||
        (path->n_points && !attributes))
        return LYG_ERR_INVALID_ARGUMENT;
    out->n_vertices = 0;
    out->n_indices = 0;
    if (path->n_verbs == 0) return LYG_OK;
    if (!check(c, hipSetDevice(c->device), "hipSetDevice")) return LYG_ERR_DEVICE;
    const size_t attr_bytes = 4ull * n_attributes * path->n_points;
    if (!ensure(c, c->in_verbs, path->n_verbs) || !ensure(c, c->in_points, 8ull * path->n_points) ||
        !ensure(c, c->in_offs, 16) || !ensure(c, c->in_opts, sizeof(lyg_stroke_options)) ||
        !ensure(c, c->in_attrs, attr_bytes) || !ensure(c, c->offs_v, 8) ||
        !ensure(c, c->offs_i, 8))
        return LYG_ERR_DEVICE;
    uint32_t* h = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(c->h_pinned) + 64);
    h[0] = 0;
    h[1] = path->n_verbs;
    h[2] = 0;
    h[3] = path->n_points;
    hipStream_t s = c->stream;
    if (!check(c, hipMemcpyAsync(c->in_verbs.p, path->verbs, path->n_verbs, hipMemcpyHostToDevice, s), "H2D") ||
        (path->n_points &&
         (!check(c, hipMemcpyAsync(c->in_points.p, path->points, 8ull * path->n_points, hipMemcpyHostToDevice, s), "H2D") ||
          !check(c, hipMemcpyAsync(c->in_attrs.p, attributes, attr_bytes, hipMemcpyHostToDevice, s), "H2D"))) ||
        !check(c, hipMemcpyAsync(c->in_offs.p, h, 16, hipMemcpyHostToDevice, s), "H2D") ||
        !check(c, hipMemcpyAsync(c->in_opts.p, opts, sizeof(*opts), hipMemcpyHostToDevice, s), "H2D"))
        return LYG_ERR_DEVICE;
    lyg::StrokeVWLaunch L{};
    L.in.verbs = as<uint8_t>(c->in_verbs);
    L.in.points = as<float>(c->in_points);
    L.in.verb_off = as<uint32_t>(c->in_offs);
    L.in.point_off = as<uint32_t>(c->in_offs) + 2;
    L.in.n_paths = 1;
    L.opts = as<lyg_stroke_options>(c->in_opts);
    L.opts_stride = 0;
    L.widths = as<float>(c->in_attrs) + width_attribute;
    L.widths_stride = n_attributes;
    L.attrs = as<float>(c->in_attrs);
    L.n_attrs = n_attributes;
    uint64_t tv = 0, ti = 0;
    std::vector<uint32_t> status;
    // a clipped miter join, or a few lines
    const bool serial =
        opts->line_join == LYG_JOIN_MITER_CLIP ||
        (path->n_points <= VW_FEW &&
         std::none_of(path->verbs, path->verbs + path->n_verbs, [](uint8_t v) {
             return v == LYG_VERB_QUADRATIC || v == LYG_VERB_CUBIC;
         }));
    int32_t st = stroke_vw_run(
        c, L, serial, out_attributes != nullptr, as<uint32_t>(c->offs_v), as<uint32_t>(c->offs_i),
        out->vertex_offset,
        [&](uint64_t nv, uint64_t ni, float** v, uint32_t** i) -> int32_t {
            if (nv > out->vertex_capacity || ni > out->index_capacity) {
                out->n_vertices = (uint32_t)nv;
                out->n_indices = (uint32_t)ni;
                return LYG_ERR_CAPACITY;
            }
            if (!ensure(c, c->out_v, 8 * nv) || !ensure(c, c->out_i, 4 * ni) ||
                (out_attributes && !ensure(c, c->out_attrs, 4ull * n_attributes * nv)))
                return LYG_ERR_DEVICE;
            L.out_attrs = out_attributes ? as<float>(c->out_attrs) : nullptr;
            *v = as<float>(c->out_v);
            *i = as<uint32_t>(c->out_i);
            return LYG_OK;
        },
        &tv, &ti, &status);
    if (st == LYG_OK) st = first_failure(status);
    if (st != LYG_OK) return st;
    if (tv && !check(c, hipMemcpy(out->vertices, c->out_v.p, 8 * tv, hipMemcpyDeviceToHost), "D2H"))
        return LYG_ERR_DEVICE;
    if (ti && !check(c, hipMemcpy(out->indices, c->out_i.p, 4 * ti, hipMemcpyDeviceToHost), "D2H"))
        return LYG_ERR_DEVICE;
    if (out_attributes && tv &&
        !check(c, hipMemcpy(out_attributes, c->out_attrs.p, 4ull * n_attributes * tv,
                            hipMemcpyDeviceToHost),
               "D2H"))
        return LYG_ERR_DEVICE;
    out->n_vertices = (uint32_t)tv;
    out->n_indices = (uint32_t)ti;
    return LYG_OK;
}

}  // extern "C"
