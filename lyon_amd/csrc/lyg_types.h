// Plain-old-data layouts shared by the host runtime and the HIP kernels.
#pragma once
#include <stdint.h>

#include "../../include/lyg.h"

namespace lyg {

// Device-side description of one batch of paths, in lyon's flat storage layout
// (path.rs:75-79): verbs[] and points[] of every path back to back, with n+1 offsets.
struct PathBatchDev {
    const uint8_t* verbs;
    const float* points;  // x, y pairs
    const uint32_t* verb_off;
    const uint32_t* point_off;
    uint32_t n_paths;
    uint32_t first_path;  // index of the first path of this launch within the batch
};

// ---- long strokes split into parts walked at once --------------------------------------
// A part of a path's walk: windows [ke, we) .. (k1, w1) of the path's steps, after a
// prologue from (k0, w0) that rebuilds the carry.  Parts of one path are walked by
// different waves; a check afterwards confirms that every part's prologue rebuilt the
// state the previous part ended in, else the path is walked again whole.
struct StrokeItem {
    uint32_t path;
    uint32_t flags;                  // ITEM_* below
    uint32_t k0, w0, ke, we, k1, w1; // verb chunk / step of the prologue, start and end
    uint32_t pt0;                    // points consumed before chunk k0
    uint32_t v_off, v_room;          // staging room (vertices), item-local ids
    uint32_t i_off, i_room;          // staging room (index slots)
    uint32_t nv, ni;                 // exact counts (vertices, index slots)
    uint32_t vbase, ibase;           // the item's first vertex / index slot in its path
};
enum : uint32_t { ITEM_FIRST = 1u, ITEM_SPLIT = 2u };
// Ids with this bit pattern (0b110 in the top three bits) refer to the first vertices of
// the path, not of the item: the last part of a split path writes them at the sub-path's
// end.  The range is apart from the item-local ids below 0x80000000 and from the stand-in
// ids the walk counts new vertices with (0x80000000 + lane << 24 + k) before their real
// ids are known: the walk compares ids for equality.
static constexpr uint32_t ID_HEAD_MARK = 0xc0000000u;
static constexpr uint32_t ID_HEAD_MASK = 0xe0000000u;
// Item-local ids start here, so the ids a part refers to in the part before it (a few
// vertices back) stay below it and far from INVALID_ID: the walk compares ids for
// equality, and an id that wrapped onto 0xffffffff would read as "no vertex".
static constexpr uint32_t ITEM_ID_BIAS = 0x40000000u;

struct F2 {
    float x, y;
};

// Per path: its first points (the first window walked alone), its items, the check.
struct StrokeHeads {
    F2 f0, f1, f2;
    uint32_t ff1, f1_base;
    uint32_t n_items, extra_first;  // item 0 is item `path`; items 1.. at extra_first..
    uint32_t redo;                  // 1: the parts disagreed or outgrew their room
};

// The carry state that decides the rest of a walk (see carry_store in stroke.hip).
struct CarryRec {
    F2 pos[3];
    F2 next[3][2];
    F2 last_kept;
    uint32_t flags[3], isp[3], code[3], base[3];
    uint32_t sp, prev_end, mnec, pad;
};

struct StrokeLaunch {
    PathBatchDev in;
    const lyg_stroke_options* opts;  // per path (opts_stride 1) or shared (stride 0)
    uint32_t opts_stride;
    // count pass outputs
    uint32_t* path_nv;
    uint32_t* path_ni;
    // emit pass inputs/outputs
    const uint32_t* vtx_off;  // exclusive offsets (n + 1)
    const uint32_t* idx_off;
    float* out_vertices;
    uint32_t* out_indices;
    uint32_t vertex_offset;  // BuffersBuilder::with_vertex_offset
    uint32_t local_ids;      // ids count from vertex_offset in every path (not the batch)
    uint32_t* work_counter;  // device work queue head (persistent kernels)
    uint32_t* err;           // emit pass: bit 0 a write outside its path's range, bit 1 a
                             // path beyond the output capacity (the path is skipped)
    uint64_t vertex_capacity;  // emit pass: output array sizes
    uint64_t index_capacity;
    const uint32_t* path_list;  // optional: the launch walks path_list[0 .. n_paths)
    uint32_t store_counts;      // emit pass also stores per-path counts (staged emit)
    const float* nsub_thr;      // round-join subdivision thresholds (31 floats) or null
    // split walks (null items: one wave walks each whole path)
    StrokeItem* items;          // n_paths + extra items; the work queue runs over n_items
    uint32_t n_items;
    // graph replay: the item count is n_paths + min(*n_extra_dev, cap_extra), and a
    // path-list walk takes its length from *n_list_dev (null: the host values above)
    const unsigned long long* n_extra_dev;
    uint32_t cap_extra;
    const uint32_t* n_list_dev;
    StrokeHeads* heads;         // per path
    CarryRec* item_spec;        // per item: the carry its prologue rebuilt
    CarryRec* item_end;         // per item: the carry at its end
};

// Staged single-pass stroke: copy of every path's staged output to its final place.
struct StrokeCompact {
    const uint32_t* path_nv;     // exact per-path counts (vertices, indices)
    const uint32_t* path_ni;
    const uint32_t* stage_voff;  // staging offsets (n + 1): the capacities' prefix sums
    const uint32_t* stage_ioff;
    const float* stage_v;
    const uint32_t* stage_i;     // path-local vertex ids
    const uint32_t* vtx_off;     // final offsets (n + 1)
    const uint32_t* idx_off;
    float* out_vertices;
    uint32_t* out_indices;
    uint32_t vertex_offset;
    uint32_t local_ids;
    uint32_t n_paths;
    uint32_t* fallback;          // paths that outgrew their staging room
    uint32_t* n_fallback;
    // split walks under graph replay: the number of items is on the device, and items
    // that would land beyond the output arrays are skipped and flagged (err bit 2)
    const unsigned long long* n_extra_dev;
    uint32_t cap_extra;
    uint64_t out_vcap, out_icap;
    uint32_t* err;
};

// Exclusive scans launched together (scan_several_kernel).
struct ScanJob {
    const uint32_t* counts;
    uint32_t n;
    uint32_t* offsets;  // n + 1
    uint64_t* total;
};
struct ScanJobs {
    ScanJob job[4];
    uint32_t n_jobs;
    uint32_t* overflow;
};

namespace fillk {
// Capacities of one wave's fill working arrays (events, heap, active edges, spans,
// monotone nodes, pending edges).
struct FillCaps {
    uint32_t ev, heap, act, span, node, below;
};
// A path's sweep that has to be done again (statuses of the sweep's own): with more room; with
// more register sets or columns of pending events than its launch had; over arrays, as it met a
// limit of every register launch.
enum : uint32_t { ST_RETRY = 100, ST_RETRY_SETS = 101, ST_RETRY_ARRAYS = 102 };
static constexpr uint32_t REG_MAX_SETS = 16;  // register sets of 64 active edges
static constexpr uint32_t REG_MAX_ROWS = 44;  // pending events per column: 66 KiB of LDS
constexpr bool is_retry(uint32_t status) { return status - ST_RETRY < 3u; }
}  // namespace fillk

// A span operation of the register sweep's log (fill_reg.hip).
struct FillOp {
    float x, y;
    uint32_t id, kind;             // vertex id; left / right vertex, begin, end
    uint32_t next;                 // the span's next operation
    uint32_t link_side, link_stack;
    uint32_t tris;                 // its triangles, then their offset in the path's
};

// A triangle of a span, until the operations' offsets are known: the nth of operation `op`.
struct FillTri {
    uint32_t a, b, c, op, nth;
};

struct FillLaunch {
    PathBatchDev in;
    const lyg_fill_options* opts;  // per path (opts_stride 1) or shared (stride 0)
    uint32_t opts_stride;
    uint8_t* work;                 // per-wave working memory (wave slot * work_stride)
    uint64_t work_stride;
    fillk::FillCaps caps;          // capacities of the per-wave arrays
    uint32_t hot_bytes;            // per-wave dynamic LDS for the hot arrays (0: none)
    uint32_t waves_per_block;
    float* stage_v;                // per-path staging, path i at stage_v_off[i] (vertices)
    uint32_t* stage_t;             // and stage_t_off[i] (triangles)
    const uint64_t* stage_v_off;
    const uint64_t* stage_t_off;
    uint32_t* path_nv;
    uint32_t* path_ni;
    uint32_t* path_status;
    uint32_t* path_round;          // the round whose staging holds the path's output
    uint32_t* path_hint;           // retry status: estimated vertices the path needs
    uint32_t round;
    const uint32_t* path_list;     // paths to process (nullptr: 0..n_list)
    uint32_t n_list;
    uint32_t* work_counter;
    uint32_t only_retry;           // only the paths whose status is retry
    // register sweep (reg_chunks 0: the sweep over arrays): sets of 64 active edges, pending
    // events per LDS column, limits below those, the log (path i's operations at
    // stage_t_off[i]) and its length per path
    uint32_t reg_chunks, heap_rows;
    uint32_t act_limit, heap_limit;
    FillOp* ops;
    FillTri* op_tris;              // as many
    uint32_t* path_ops;
    // copy pass
    const uint32_t* vtx_off;
    const uint32_t* idx_off;
    float* out_vertices;
    uint32_t* out_indices;
    uint32_t vertex_offset;
    uint32_t local_ids;            // ids count from vertex_offset in every path
    // output capacity (vertices, indices): a path whose range ends past it is not copied
    uint64_t vertex_capacity;
    uint64_t index_capacity;
};

// Variable-width stroke (stroke_vw_kernel): one lane per path, count then emit.
struct StrokeVWLaunch {
    PathBatchDev in;
    const lyg_stroke_options* opts;
    uint32_t opts_stride;
    const float* widths;     // per point of the batch: the width factor of its endpoint
    uint32_t widths_stride;  // floats per point (custom attributes per endpoint)
    uint32_t* path_nv;       // count pass
    uint32_t* path_ni;
    uint32_t* path_status;
    const uint32_t* vtx_off;  // emit pass
    const uint32_t* idx_off;
    float* out_vertices;
    uint32_t* out_indices;
    uint32_t vertex_offset;
    uint32_t* err;
    uint32_t paths_per_wave;  // lanes of a wave that take paths (1-64); the rest idle
    // optional: every vertex's interpolated custom attributes (n_attrs per vertex) from the
    // attribute table (n_attrs per point of the batch)
    const float* attrs;
    uint32_t n_attrs;
    float* out_attrs;
    // the paths to walk: list[0 .. *n_list) (null: all)
    const uint32_t* list;
    const uint32_t* n_list;
};

// Joins per window of the parallel variable-width stroke.
static constexpr uint32_t VW_WINDOW = 63u;
// The end of a sub-path of the parallel variable-width stroke.
struct VWTail {
    uint32_t path, first, count;  // its points: first .. first + count of the path's kept ones
    uint32_t flags;               // 1: closed, 2: a point was dropped after the first
    uint32_t nv, nt;              // what its end emits
    // set by the emit pass, in vertices / triangles of the path: where its end starts, the
    // first vertices of the joins at its second and at its last but one buffered point
    uint32_t v_at, t_at, f1_base, p_base;
};
// Parallel variable-width stroke (stroke_vw.hip).
struct VWPar {
    PathBatchDev in;
    const lyg_stroke_options* opts;
    uint32_t opts_stride;
    const float* widths;
    uint32_t widths_stride;
    const float* attrs;
    uint32_t n_attrs;
    float* out_attrs;
    // per path: the plan's counts and their offsets (n + 1), the kept points, 0 parallel /
    // 1 serial / 2 nothing to walk, and the results
    uint32_t *raw_n, *win_n, *tail_n, *att_cap_n;
    const uint32_t *raw_off, *win_off, *tail_off, *att_off;
    uint32_t *kept_n, *path_mode, *path_status, *path_nv, *path_ni;
    // per kept point (a path's at raw_off): x, y, half width, running length; flags; vertex
    // source (null without vertex attributes)
    float* rec;
    uint8_t* pflags;
    float* src_t;
    uint32_t* src_id;
    // edges with side lines (a path's at att_off): point (~0: unused slot), four floats
    uint32_t* att_point;
    float* att_n;
    // per window
    uint32_t *win_att, *win_nv, *win_ni;
    const uint32_t *win_voff, *win_ioff;
    uint32_t n_windows;
    VWTail* tails;
    uint32_t n_tails;
    uint32_t *slow_list, *cands, *dirty;
    uint32_t cand_cap, dirty_cap;
    // [1] serial paths, [2] candidates, [3] windows to count
    // again, [4] a list overflowed, [5] some path has more than `few` points
    uint32_t* ctr;
    uint32_t few;
    const uint32_t *vtx_off, *idx_off;
    float* out_vertices;
    uint32_t* out_indices;
    uint32_t vertex_offset;
    uint32_t* err;
};

struct FlattenLaunch {
    const int32_t* kinds;  // 0 line, 1 quadratic, 2 cubic
    const float* ctrl;     // 8 floats per segment: from, ctrl1, ctrl2, to
    uint32_t n;
    float tolerance;
    uint32_t* counts;         // count pass
    const uint32_t* offsets;  // emit pass (n + 1)
    float* out_points;
    uint32_t* runs;           // per run of 16 output points: segment, t bits (null: the emit
                              // searches the offsets and computes t)
    float* polys;             // with runs: 12 floats per segment (polynomial form, step, n)
};

// Path validators (lyon_algorithms hit_test.rs / area.rs) over the batched layout.
struct ValidateLaunch {
    const uint8_t* verbs;
    const float* points;
    const uint32_t* verb_off;   // n_paths + 1
    const uint32_t* point_off;  // n_paths + 1
    uint32_t n_paths;
    float tolerance;
    // winding numbers: one query point per entry, against path query_path[i]
    const float* queries;  // x, y pairs
    const uint32_t* query_path;
    uint32_t n_queries;
    int fill_rule;          // 0 EvenOdd, 1 NonZero (for `inside`)
    int32_t* winding;       // n_queries
    uint8_t* inside;        // n_queries or null
    // areas: one per path
    float* areas;
};

// SVG path data parse (svg.hip): a wave per string, or a lane.
struct SvgLaunch {
    const uint8_t* text;
    const uint32_t* text_off;  // n + 1
    uint32_t n;
    int num_attributes;
    int stop_at;               // ASCII character or -1
    uint32_t* counts_v;
    uint32_t* counts_p;
    int32_t* errors;           // 4 per string or null
    uint32_t* n_errors;        // [0] strings with an error, [1] staging rooms overflowed
    uint8_t* verbs;            // staging rooms (see svg_parse_kernel)
    float* points;
    uint32_t by_wave;          // a wave per string first; counts_v: SVG_LEFT for the serial parser
    // compaction
    const uint32_t* off_v;
    const uint32_t* off_p;
};

}  // namespace lyg
