"""GPU parity of the fill tessellator (plain and batched) against the oracle.

Bar, per path:
  * the same status (where lyon panics — a Rust index out of bounds or unreachable!() in
    its sweep, reachable only without intersection handling — the GPU returns
    InternalError);
  * vertices bit-exact and in the same order;
  * the same set of triangles (each rotated to start at its smallest id; lyon writes a
    span's triangles when the span ends, the GPU as they form, so only the order in the
    index buffer differs);
  * per-sample coverage identical on a 4096 x 4096 grid over the path (samples within 1e-4
    of a triangle edge excluded) and total area within 1e-6 relative.
"""
import numpy as np
import pytest

from helpers import FILL_KATS, bbox_diag, fill_corpus
from lyon_amd import BuffersBuilder, FillOptions, FillRule, FillTessellator, VertexBuffers
from lyon_amd import workloads
from lyon_amd.path import Path, PathBuilder, polygon
from lyon_amd.tessellation import Orientation, TessellationError
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

PANIC = 6      # oracle status: the reference panics
INTERNAL = 5   # TessellationError::Internal


def gpu_fill(path, opts, vertex_offset=0):
    buf = VertexBuffers()
    try:
        FillTessellator().tessellate_path(path, opts,
                                          BuffersBuilder(buf).with_vertex_offset(vertex_offset))
    except TessellationError as e:
        return e.code, None, None
    return 0, buf.vertices, buf.indices


def ref_fill(path, opts, vertex_offset=0):
    return O.fill(path, opts.tolerance, int(opts.fill_rule), int(opts.sweep_orientation),
                  opts.handle_intersections, vertex_offset)


def canon(idx):
    t = np.asarray(idx, np.int64).reshape(-1, 3)
    if len(t) == 0:
        return t
    k = np.argmin(t, axis=1)
    r = np.arange(len(t))
    t = np.stack([t[r, k], t[r, (k + 1) % 3], t[r, (k + 2) % 3]], 1)
    return t[np.lexsort(t.T[::-1])]


def check(path, opts, what, coverage=True, vertex_offset=0):
    gst, gv, gi = gpu_fill(path, opts, vertex_offset)
    rst, rv, ri = ref_fill(path, opts, vertex_offset)
    if rst == PANIC:
        assert gst == INTERNAL, f"{what}: reference panics, gpu status {gst}"
        return
    assert gst == rst, f"{what}: status gpu {gst} != reference {rst}"
    if rst != 0:
        return
    assert len(gv) == len(rv), f"{what}: {len(gv)} vertices != {len(rv)}"
    assert np.array_equal(np.asarray(gv, np.float32).view(np.uint32),
                          np.asarray(rv, np.float32).view(np.uint32)), f"{what}: vertices differ"
    assert len(gi) == len(ri), f"{what}: {len(gi) // 3} triangles != {len(ri) // 3}"
    assert np.array_equal(canon(gi), canon(ri)), f"{what}: triangle sets differ"
    if coverage and len(ri):
        lv = np.asarray(gv, np.float32)
        c = O.coverage_compare(rv, np.asarray(ri, np.int64) - vertex_offset, lv,
                               np.asarray(gi, np.int64) - vertex_offset, n=4096, eps=1e-4)
        assert c["mismatch"] == 0, f"{what}: {c['mismatch']} samples differ"
        rel = abs(c["area_a"] - c["area_b"]) / max(c["area_a"], 1e-300)
        assert rel <= 1e-6, f"{what}: area differs by {rel}"


OPTION_SETS = {
    "evenodd": FillOptions(tolerance=0.05, fill_rule=FillRule.EvenOdd),
    "nonzero": FillOptions(tolerance=0.05, fill_rule=FillRule.NonZero),
    "horizontal": FillOptions(tolerance=0.1, fill_rule=FillRule.EvenOdd,
                              sweep_orientation=Orientation.Horizontal),
    "no_intersections": FillOptions(tolerance=0.05, fill_rule=FillRule.NonZero,
                                    handle_intersections=False),
}

CORPUS = fill_corpus()


@pytest.mark.parametrize("opt_name", list(OPTION_SETS))
def test_corpus(opt_name):
    """KAT polygons, lyon's fuzz and earcut fixtures, the plain workload path, stars."""
    opts = OPTION_SETS[opt_name]
    for k, (name, p) in enumerate(CORPUS):
        print(f"{opt_name} {name}", flush=True)
        check(p, opts, f"{opt_name}/{name}", coverage=(opt_name == "evenodd"),
              vertex_offset=7 * k)


@pytest.mark.parametrize("name,pts,step,expected", FILL_KATS, ids=[k[0] for k in FILL_KATS])
def test_kat_rotations(name, pts, step, expected):
    """fill_tests.rs triangle counts under rotation (every 0.05 rad)."""
    base = polygon(pts, True)
    for a in np.arange(0.0, 2 * np.pi, 0.05, dtype=np.float32):
        c, s = np.cos(a), np.sin(a)
        pp = base.points @ np.array([[c, s], [-s, c]], np.float32)
        path = Path(base.verbs, pp.astype(np.float32))
        st, v, i = gpu_fill(path, FillOptions(tolerance=0.05))
        assert st == 0
        rst, rv, ri = ref_fill(path, FillOptions(tolerance=0.05))
        assert len(i) // 3 == len(ri) // 3, f"{name} at {a}"
        check(path, FillOptions(tolerance=0.05, fill_rule=FillRule.NonZero), f"{name}@{a}",
              coverage=False)


def test_errors_and_empty():
    p = polygon([(0, 0), (1, 1), (0, 1)], True)
    for t in (0.0, -1.0, float("nan")):
        st, _, _ = gpu_fill(p, FillOptions(tolerance=t))
        assert st == 4  # UnsupportedParamater::ToleranceIsNaN
    empty = Path(np.zeros(0, np.uint8), np.zeros((0, 2), np.float32))
    st, v, i = gpu_fill(empty, FillOptions())
    assert st == 0 and len(v) == 0 and len(i) == 0
    b = PathBuilder(); b.begin((0, 0)); b.line_to((float("nan"), 1)); b.line_to((1, 1)); b.end(True)
    st, _, _ = gpu_fill(b.build(), FillOptions())
    assert st == 3  # UnsupportedParamater::PositionIsNaN


def test_curves_and_vertex_offset():
    """Curved paths (the plain workload and cubic loops) at several tolerances."""
    batch = workloads.fill_batch(16, seed=3)
    for i in range(len(batch)):
        for tol in (0.5, 0.05):
            check(batch.path(i), FillOptions(tolerance=tol, fill_rule=FillRule(i % 2)),
                  f"fill_batch[{i}] tol {tol}", coverage=(i < 4), vertex_offset=1000 * i)


def test_batch_matches_plain_calls():
    """The batched form equals tessellate_path per path into one shared VertexBuffers."""
    from lyon_amd.batch import DeviceBatch, FillBatcher
    n = 192
    batch = workloads.fill_batch(n, seed=0)
    opts = workloads.fill_options(n, tolerance=0.05)
    res = FillBatcher().run(DeviceBatch(batch, opts), vertex_offset=5)
    vo = res.vertex_offsets
    status = res.status
    allv = res.all_vertices()
    alli = res.all_indices()
    io = res.index_offsets
    for i in range(n):
        o = FillOptions(tolerance=0.05, fill_rule=FillRule(int(opts[i]["fill_rule"])))
        rst, rv, ri = ref_fill(batch.path(i), o, vertex_offset=5 + int(vo[i]))
        assert status[i] == rst, f"path {i}: status {status[i]} != {rst}"
        gv = allv[vo[i]:vo[i + 1]]
        gi = alli[io[i]:io[i + 1]]
        assert np.array_equal(gv.view(np.uint32), np.asarray(rv, np.float32).view(np.uint32)), \
            f"batch path {i}: vertices differ"
        assert np.array_equal(canon(gi), canon(ri)), f"batch path {i}: triangle sets differ"


def test_lds_resident_form_and_fallback():
    """The batched fill gives the same bytes whether its first round keeps each path's active
    edges in registers (the default), sweeps over arrays that start in LDS and move to global
    memory as they grow, or keeps them in registers at an eighth of the estimated capacities (so
    that many paths outgrow them and are swept again over arrays); paths of every size of the
    fill workload, the 513-point stars included."""
    from lyon_amd.batch import DeviceBatch, FillBatcher, set_fill_lds_resident, synchronize
    n = 512
    batch = workloads.fill_batch(n, seed=0)
    opts = workloads.fill_options(n, tolerance=0.05)
    db = DeviceBatch(batch, opts)
    outs = []
    try:
        for mode in (1, 0, 8):
            set_fill_lds_resident(mode)
            res = FillBatcher().run(db)
            synchronize()
            outs.append((mode, res.status.copy(), res.all_vertices().copy(),
                         res.all_indices().copy()))
    finally:
        set_fill_lds_resident(True)
    m0, st0, v0, i0 = outs[0]
    assert np.all(st0 == 0)
    for m, st, v, i in outs[1:]:
        assert np.array_equal(st, st0), f"mode {m}: statuses differ"
        assert np.array_equal(v.view(np.uint32), v0.view(np.uint32)), f"mode {m}: vertices differ"
        assert np.array_equal(i, i0), f"mode {m}: indices differ"


def test_many_launches_in_one_round():
    """Paths in many size classes and forms (fill-workload stars and cubic loops, closed random
    walks of 2,000 to 60,000 vertices) give a round about ten launches (a host-side test plans
    all 32): every path is swept (status 0) and the bytes equal those of the sweep over
    arrays."""
    from lyon_amd.batch import DeviceBatch, FillBatcher, set_fill_lds_resident, synchronize
    from lyon_amd.path import PathBatch
    base = workloads.fill_batch(1024, seed=2)
    paths = [base.path(i) for i in range(len(base))]
    for k, nv in enumerate((2000, 7000, 20000, 60000)):
        paths.append(workloads.random_walk_path(nv, seed=k + 1, extent=4096.0))
    batch = PathBatch.from_paths(paths)
    opts = workloads.fill_options(len(paths), tolerance=0.05, seed=3)
    db = DeviceBatch(batch, opts)
    outs = []
    try:
        for mode in (1, 0):
            set_fill_lds_resident(mode)
            res = FillBatcher().run(db)
            synchronize()
            outs.append((res.status.copy(), res.all_vertices().copy(), res.all_indices().copy()))
    finally:
        set_fill_lds_resident(True)
    (s1, v1, i1), (s0, v0, i0) = outs
    assert np.all(s1 == 0) and np.array_equal(s1, s0)
    assert np.array_equal(v1.view(np.uint32), v0.view(np.uint32))
    assert np.array_equal(i1, i0)


def zigzag(edges):
    """A closed comb: a horizontal line crosses up to `edges` of its edges."""
    n = edges // 2
    pts = []
    for i in range(n):
        pts += [(float(4 * i), 0.25 * (i % 7)), (float(4 * i + 1), 1000.0 + 0.5 * (i % 5))]
    return polygon(pts + [(4.0 * n, 0.0), (4.0 * n, 1010.0), (-2.0, 1010.0), (-2.0, 0.0)])


def fan(edges):
    """Thin triangles with one apex on top: `edges` edges start at one point."""
    b = PathBuilder()
    for i in range(edges // 2):
        b.begin((0.0, 0.0))
        b.line_to((20.0 * i - 300.0, 500.0))
        b.line_to((20.0 * i - 290.0, 500.0 + i % 3))
        b.end(True)
    return b.build()


@pytest.mark.parametrize("shape,sizes", [
    (zigzag, (118, 122, 124, 126, 128, 130)),          # 2 sets of 64 active edges
    (zigzag, (310, 314, 316, 318, 320, 322)),          # 5 sets
    (zigzag, (1014, 1018, 1020, 1022, 1024, 1026, 1830, 1900, 2100)),  # 16 sets; beyond
    (fan, (60, 62, 64, 66, 126, 128, 130)),            # 64 edges below one event
], ids=["two_sets", "five_sets", "sixteen_sets", "edges_below"])
def test_active_edges_around_the_register_sets(shape, sizes):
    """Paths whose active edges, or edges below one event, just fit the register sweep or
    just outgrow it: plain calls, a batch and a captured batch all give the oracle's
    vertices and triangles."""
    from lyon_amd.batch import DeviceBatch, FillBatcher, FillGraph, synchronize
    from lyon_amd.path import PathBatch
    paths = [shape(k) for k in sizes]
    o = FillOptions(tolerance=0.05)
    refs = [ref_fill(p, o) for p in paths]
    for k, p in zip(sizes, paths):
        check(p, o, f"{shape.__name__} {k}", coverage=False)
    opts = workloads.fill_options(len(paths), tolerance=0.05)
    opts["fill_rule"] = int(o.fill_rule)
    db = DeviceBatch(PathBatch.from_paths(paths), opts)
    res = FillBatcher().run(db)
    synchronize()
    graph = FillGraph(db, int(res.n_vertices), int(res.n_indices))
    graph.launch()
    for r in (res, graph.result()):
        v, i, vo, io = r.all_vertices(), r.all_indices(), r.vertex_offsets, r.index_offsets
        for k, (st, rv, ri) in enumerate(refs):
            assert r.status[k] == st == 0
            assert np.array_equal(v[vo[k]:vo[k + 1]].view(np.uint32),
                                  np.asarray(rv, np.float32).view(np.uint32)), sizes[k]
            assert np.array_equal(canon(i[io[k]:io[k + 1]]),
                                  canon(np.asarray(ri, np.int64) + int(vo[k]))), sizes[k]


@pytest.mark.parametrize("sizes", [(1, 2, 3, 62, 63, 64, 65), (1021, 1022, 1023, 1024),
                                   (3, 4093, 4094, 4095, 4096)], ids=["few", "1024", "4096"])
def test_paths_around_the_verbs_measured_at_once(sizes):
    """Paths of as many verbs as are measured together (64 a turn, boxes of 1,024, of 4,096
    again, none beyond), closed outlines that cross themselves here and there."""
    from lyon_amd.batch import DeviceBatch, FillBatcher
    from lyon_amd.path import PathBatch
    rng = np.random.default_rng(sizes[0])
    paths = []
    for n in sizes:  # n + 1 verbs: Begin, lines and curves, Close
        b = PathBuilder()
        t = np.arange(n) * (2.0 * np.pi / max(n, 1))
        r = 400.0 + 40.0 * np.sin(7.0 * t) + rng.random(n)
        p = np.stack([r * np.cos(t), r * np.sin(2.0 * t)], 1)
        b.begin(tuple(p[0]))
        for k in range(1, n):
            m = tuple((p[k - 1] + p[k]) * 0.5 + 0.5)
            if k % 5 == 1:
                b.quadratic_bezier_to(m, tuple(p[k]))
            elif k % 5 == 2:
                b.cubic_bezier_to(tuple(p[k - 1]), m, tuple(p[k]))
            else:
                b.line_to(tuple(p[k]))
        b.end(True)
        paths.append(b.build())
    opts = workloads.fill_options(len(paths), tolerance=0.05)
    res = FillBatcher().run(DeviceBatch(PathBatch.from_paths(paths), opts))
    v, i, vo, io = res.all_vertices(), res.all_indices(), res.vertex_offsets, res.index_offsets
    for k, p in enumerate(paths):
        o = FillOptions(tolerance=0.05, fill_rule=FillRule(int(opts[k]["fill_rule"])))
        st, rv, ri = ref_fill(p, o, int(vo[k]))
        assert res.status[k] == st == 0
        assert np.array_equal(v[vo[k]:vo[k + 1]].view(np.uint32),
                              np.asarray(rv, np.float32).reshape(-1, 2).view(np.uint32)), sizes[k]
        assert np.array_equal(canon(i[io[k]:io[k + 1]]), canon(ri)), sizes[k]


def test_very_large_path():
    """fill_tests.rs:2140-2166: a path of 1,000,000 endpoints (two wiggling sides of a long
    band) fills without error; the same vertices and triangle count as the oracle and the
    same area."""
    from lyon_amd import PathBuilder
    n = 1_000_000
    d = np.float32(0.0)
    step = np.float32(0.1)
    pts = np.zeros((n, 2), np.float32)
    for k in range(n // 2):
        pts[k] = (np.cos(d, dtype=np.float32), d)
        d = np.float32(d + step)
    for k in range(n // 2, n):
        pts[k] = (np.float32(np.cos(d, dtype=np.float32) + np.float32(30.0)), d)
        d = np.float32(d - step)
    b = PathBuilder()
    b.begin((0.0, 0.0))
    for p in pts:
        b.line_to(p)
    b.end(True)
    path = b.build()
    vb = VertexBuffers()
    FillTessellator().tessellate_path(path, FillOptions(), BuffersBuilder(vb))
    st, rv, ri = O.fill(path, 0.1, 0)
    assert st == 0
    assert len(vb.vertices) == len(rv) and len(vb.indices) == len(ri)
    c = O.coverage_compare(rv, ri, vb.vertices, vb.indices, n=256)
    assert c["mismatch"] == 0 and abs(c["area_a"] - c["area_b"]) <= 1e-6 * c["area_b"]


def test_without_memory_for_the_span_log():
    """Where the register sweep's log (52 bytes per staged triangle) cannot be allocated, the
    paths are swept over arrays, which need none: an eager call and a captured one on a context
    that refuses the log give the bytes of one that does not.  20,000 triangles stage 12
    million: 388 MB of the log's larger array, 146 MB of triangles."""
    import ctypes as C
    import threading

    from lyon_amd import _lib
    from lyon_amd.batch import DeviceBatch, FillBatcher, FillGraph, _Ctx, synchronize
    from lyon_amd.path import PathBatch
    rng = np.random.default_rng(9)
    n = 20000
    batch = PathBatch.from_paths([polygon(t) for t in rng.uniform(0, 500, (n, 3, 2))])
    db = DeviceBatch(batch, workloads.fill_options(n, tolerance=0.05))
    lib = C.CDLL(_lib.LIB_PATH)
    lib.lyg_ctx_set_alloc_limit.argtypes = [C.c_void_p, C.c_uint64]
    lib.lyg_ctx_set_alloc_limit.restype = None
    outs = {}

    def fresh(limit):  # a context of its own
        lib.lyg_ctx_set_alloc_limit(_Ctx.get(), limit)
        res = FillBatcher().run(db)
        said = _lib.lib().lyg_ctx_last_error(_Ctx.get()).decode()
        synchronize()
        g = FillGraph(db, int(res.n_vertices), int(res.n_indices))
        g.launch()
        outs[limit] = [said] + [(r.status.copy(), r.all_vertices().view(np.uint32).copy(),
                                 r.all_indices().copy()) for r in (res, g.result())]

    for limit in (0, 256 << 20):
        t = threading.Thread(target=fresh, args=(limit,))
        t.start()
        t.join()
    assert "limit" not in outs[0][0] and "limit" in outs[256 << 20][0]
    first = outs[0][1]
    assert not first[0].any() and len(first[1]) > 0
    for other in outs[0][2:] + outs[256 << 20][1:]:
        assert all(np.array_equal(a, b) for a, b in zip(first, other))


@pytest.mark.parametrize("shape,size,rounds", [
    (fan, 62, 1), (fan, 126, 2),             # more than 64 edges below one event: over arrays next
    (zigzag, 126, 1), (zigzag, 1900, 1),     # estimated right; below, counted
    (zigzag, 1020, 1), (zigzag, 1100, 1), (zigzag, 1500, 1), (zigzag, 1790, 1)],
    ids=["fan62", "fan126", "zigzag126", "zigzag1900", "zigzag1020", "zigzag1100", "zigzag1500",
         "zigzag1790"])
def test_rounds_of_paths_that_outgrow_the_registers(shape, size, rounds):
    """A path that meets a limit of every register launch is swept over arrays in the next
    round, with the room it had (it needed no more).  A comb's edges are all active at once,
    twice what half the degrees say: where that is beyond the registers it is known before, in
    both orientations."""
    import ctypes as C

    from lyon_amd import _lib
    from lyon_amd.batch import _Ctx
    up, side = shape(size), shape(size)
    side.points = np.stack([side.points[:, 1], -side.points[:, 0]], axis=1)
    for path, way in ((up, Orientation.Vertical), (side, Orientation.Horizontal)):
        st, _, _ = gpu_fill(path, FillOptions(tolerance=0.05, sweep_orientation=way))
        n, scale = C.c_uint32(0), C.c_uint64(0)
        C.CDLL(_lib.LIB_PATH).lyg_ctx_last_fill(C.c_void_p(_Ctx.get()), C.byref(n),
                                                C.byref(scale))
        assert st == 0 and (n.value, scale.value) == (rounds, 1)
