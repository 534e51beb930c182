"""Variable-width stroke (StrokeOptions::variable_line_width) on the GPU against the oracle
(stroke.rs:653-767, 1380-1512, 1809-1866, 2060-2128), through lyg_stroke_path_vw and
lyg_stroke_batch_vw.

Tolerance: the same triangles (index triples) and positions within 1e-4 of the path's
scale (max |coordinate|, at least 1) -- the edge normals go through asin, cos and sin,
evaluated in f64 and rounded once on the GPU and by the C library on the CPU, which may
differ in the last bit.  NaN positions (lyon's own, at sharp turns inside cubics) must be
NaN on both sides.  On random paths a near-tie decided differently by one bit may change a
join's layout: at least 97% of the paths must match exactly, and every path must have the
same status."""
import numpy as np
import pytest

from helpers import counted_curves
from lyon_amd import (BuffersBuilder, LineCap, LineJoin, StrokeOptions, StrokeTessellator,
                      VertexBuffers)
from lyon_amd import workloads
from lyon_amd.batch import DeviceBatch, StrokeVWBatcher, synchronize
from lyon_amd.path import PathBuilder
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


def gpu_vw(path, opts):
    buf = VertexBuffers()
    StrokeTessellator().tessellate_path(path, opts, BuffersBuilder(buf))
    return np.asarray(buf.vertices, np.float32).reshape(-1, 2), np.asarray(buf.indices)


def ref_vw(path, opts):
    st, v, i = O.stroke(path, line_width=opts.line_width, miter_limit=opts.miter_limit,
                        tolerance=opts.tolerance, start_cap=int(opts.start_cap),
                        end_cap=int(opts.end_cap), line_join=int(opts.line_join),
                        widths=path.attributes[:, opts.variable_line_width])
    assert st == 0
    return v, i


def close_enough(v, rv, scale):
    if v.shape != rv.shape:
        return False
    nan_a, nan_b = np.isnan(v), np.isnan(rv)
    if not np.array_equal(nan_a, nan_b):
        return False
    ok = ~nan_a
    return bool(np.all(np.abs(v[ok] - rv[ok]) <= 1e-4 * scale))


def square_path():
    b = PathBuilder(1)
    for pts in (((-1, 1), (1, 1), (1, -1), (-1, -1)), ((-1, -1), (1, -1), (1, 1), (-1, 1))):
        b.begin(pts[0], [0.3])
        for q in pts[1:]:
            b.line_to(q, [0.3])
        b.end(False)
    return b.build()


def issue_894_path():
    b = PathBuilder(1)
    b.begin((435.72, 368.42), [38.82])
    b.line_to((433.53, 366.06), [38.82])
    b.quadratic_bezier_to((431.35, 363.70), (430.22, 362.52), [39.59])
    b.quadratic_bezier_to((429.09, 361.34), (429.05, 362.14), [41.62])
    b.line_to((429.00, 362.95), [41.63])
    b.end(False)
    return b.build()


def growing_spiral():
    """Curves and lines whose width factor grows along the path (0.2 to 3), closed."""
    b = PathBuilder(2)
    b.begin((0, 0), [9.0, 0.2])
    b.quadratic_bezier_to((50, -40), (100, 0), [9.0, 0.8])
    b.cubic_bezier_to((140, 40), (60, 120), (20, 80), [9.0, 1.6])
    b.line_to((-30, 60), [9.0, 2.2])
    b.line_to((-10, 10), [9.0, 3.0])
    b.end(True)
    return b.build()


@pytest.mark.parametrize("case", ["square", "issue_894", "spiral"])
@pytest.mark.parametrize("join", [LineJoin.Miter, LineJoin.MiterClip, LineJoin.Round,
                                  LineJoin.Bevel])
@pytest.mark.parametrize("cap", [LineCap.Butt, LineCap.Square, LineCap.Round])
def test_plain_calls_match_the_oracle(case, join, cap):
    path = {"square": square_path, "issue_894": issue_894_path, "spiral": growing_spiral}[case]()
    attr = 1 if case == "spiral" else 0
    opts = StrokeOptions(line_width=2.0 if case == "spiral" else 1.0, line_join=join,
                         start_cap=cap, end_cap=cap, miter_limit=2.0, tolerance=0.01,
                         variable_line_width=attr)
    v, i = gpu_vw(path, opts)
    rv, ri = ref_vw(path, opts)
    if case == "square" and join == LineJoin.Miter and cap == LineCap.Butt:
        assert len(i) // 3 == 12  # test_square (stroke.rs:2851-2908)
    if case == "square" and join == LineJoin.Bevel and cap == LineCap.Square:
        assert len(i) // 3 == 16
    assert np.array_equal(i, ri)
    scale = max(1.0, float(np.max(np.abs(path.points))))
    assert close_enough(v, rv, scale)


def test_empty_caps():
    """test_empty_caps (stroke.rs:2918-2976): none with butt caps, 8 triangles with square
    caps, the oracle's bytes with round caps."""
    b = PathBuilder(1)
    b.begin((1, 0), [1.0]); b.end(True)
    b.begin((2, 0), [1.0]); b.line_to((2, 0), [1.0]); b.end(False)
    b.begin((3, 0), [1.0]); b.line_to((3, 0), [1.0]); b.end(True)
    b.begin((3, 0), [1.0])
    for _ in range(3):
        b.line_to((3, 0), [1.0])
    b.end(True)
    b.begin((4, 0), [1.0]); b.end(False)
    p = b.build()
    for cap, want in ((LineCap.Butt, 0), (LineCap.Square, 8), (LineCap.Round, None)):
        opts = StrokeOptions(start_cap=cap, end_cap=cap, variable_line_width=0)
        v, i = gpu_vw(p, opts)
        rv, ri = ref_vw(p, opts)
        if want is not None:
            assert len(i) // 3 == want
        assert np.array_equal(i, ri) and close_enough(v, rv, 4.0)


def random_batch(n, seed):
    batch = workloads.stroke_batch(n, 4, 48, 1024.0, seed=seed)
    opts = workloads.stroke_options(n, tolerance=0.05, seed=seed)
    rng = np.random.default_rng(seed)
    widths = rng.uniform(0.25, 2.5, len(batch.points)).astype(np.float32)
    return batch, opts, widths


@pytest.mark.parametrize("seed", [1, 2])
def test_batch_matches_the_oracle(seed):
    n = 400
    batch, opts, widths = random_batch(n, seed)
    db = DeviceBatch(batch, opts)
    res = StrokeVWBatcher(widths).run(db, vertex_offset=7, check=False)
    synchronize()
    st = res.status
    vo, io = res.vertex_offsets, res.index_offsets
    v, i = res.all_vertices(), res.all_indices()
    exact = 0
    for p in range(n):
        path = batch.path(p)
        o = opts[p]
        pb, pe = int(batch.point_offsets[p]), int(batch.point_offsets[p + 1])
        rs, rv, ri = O.stroke(path, line_width=float(o["line_width"]),
                              miter_limit=float(o["miter_limit"]),
                              tolerance=float(o["tolerance"]), start_cap=int(o["start_cap"]),
                              end_cap=int(o["end_cap"]), line_join=int(o["line_join"]),
                              vertex_offset=7 + int(vo[p]), widths=widths[pb:pe])
        assert int(st[p]) == rs
        pv = v[vo[p]:vo[p + 1]]
        pi = i[io[p]:io[p + 1]]
        scale = max(1.0, float(np.max(np.abs(path.points))))
        if np.array_equal(pi, ri) and close_enough(pv, rv, scale):
            exact += 1
    print(f"{exact} of {n} paths match exactly", flush=True)
    assert exact >= 0.97 * n


@pytest.mark.parametrize("join", [LineJoin.Miter, LineJoin.MiterClip, LineJoin.Round])
@pytest.mark.parametrize("closed", [False, True])
def test_sub_paths_around_the_window_size(join, closed):
    """Sub-paths of 1-5, 61-66 and 125-129 points (a window holds 63 joins and repeats the
    one before), one per path and several in a path, with repeated points that are dropped,
    and curves whose joins may fold back (widths that change by more than an edge)."""
    rng = np.random.default_rng(9)
    paths = []
    for counts in ([1], [2], [3], [4], [5], [61], [62], [63], [64], [65], [66], [125], [126],
                   [127], [128], [129], [62, 1, 64], [63, 63, 2], [5, 126, 3]):
        b = PathBuilder(1)
        for k in counts:
            pts = rng.uniform(0, 300, (k, 2)).round(1)
            b.begin(tuple(pts[0]), [rng.uniform(0.2, 2)])
            for q in pts[1:]:
                b.line_to(tuple(q), [rng.uniform(0.2, 2)])
                if rng.random() < 0.1:
                    b.line_to(tuple(q), [1.0])
            b.end(closed)
        paths.append(b.build())
    for _ in range(60):
        b = PathBuilder(1)
        b.begin((0, 0), [1.0])
        for _ in range(8):
            b.cubic_bezier_to(*[tuple(q) for q in rng.uniform(0, 60, (3, 2))],
                              [rng.uniform(0.2, 12)])
        b.end(closed)
        paths.append(b.build())
    same = 0
    for path in paths:
        opts = StrokeOptions(line_width=2.0, line_join=join, start_cap=LineCap.Round,
                             end_cap=LineCap.Square, tolerance=0.05, variable_line_width=0)
        v, i = gpu_vw(path, opts)
        rv, ri = ref_vw(path, opts)
        same += np.array_equal(i, ri) and close_enough(v, rv, 300.0)
    assert same >= 0.97 * len(paths), same
    o = vw_options(len(paths), rng, 2.0, 0.05)
    o["line_join"] = int(join)
    serial, _ = forms(paths, o)
    assert serial == len(paths) if join == LineJoin.MiterClip else serial < len(paths) // 4


@pytest.mark.parametrize("counts", [[1, 2, 15, 16, 17, 18], [31, 33, 63, 65, 80], [4000, 90, 70],
                                    [4080, 16, 50], [4095, 4097], [64, 9000, 20]])
def test_curves_around_the_listed_steps(counts):
    """Curves of as many points as the t of every 16th of 4,096 steps is listed for, starting
    and ending around those numbers."""
    rng = np.random.default_rng(counts[0])
    tol = 1e-2
    opts = StrokeOptions(line_width=1.0, line_join=LineJoin.Miter, tolerance=tol,
                         variable_line_width=0)
    for shift in (0, 1, 15):
        b = PathBuilder(1)
        counted_curves(b, [3] * shift + counts, tol, rng, lambda: [rng.uniform(0.5, 2.0)])
        b.end(shift == 1)
        path = b.build()
        v, i = gpu_vw(path, opts)
        rv, ri = ref_vw(path, opts)
        assert np.array_equal(i, ri), shift
        assert close_enough(v, rv, float(np.ptp(np.asarray(path.points), axis=0).max())), shift


def test_batch_equals_plain_calls():
    n = 24
    batch, opts, widths = random_batch(n, 3)
    db = DeviceBatch(batch, opts)
    res = StrokeVWBatcher(widths).run(db, check=False)
    vo, io = res.vertex_offsets, res.index_offsets
    v, i = res.all_vertices(), res.all_indices()
    for p in range(n):
        o = opts[p]
        pb, pe = int(batch.point_offsets[p]), int(batch.point_offsets[p + 1])
        path = batch.path(p)
        path.attributes = widths[pb:pe].reshape(-1, 1)
        so = StrokeOptions(line_width=float(o["line_width"]), miter_limit=float(o["miter_limit"]),
                           tolerance=float(o["tolerance"]), start_cap=int(o["start_cap"]),
                           end_cap=int(o["end_cap"]), line_join=int(o["line_join"]),
                           variable_line_width=0)
        gv, gi = gpu_vw(path, so)
        assert np.array_equal(gv.view(np.uint32), v[vo[p]:vo[p + 1]].view(np.uint32))
        assert np.array_equal(gi.astype(np.int64) + int(vo[p]), i[io[p]:io[p + 1]])


def test_vertex_attributes_match_the_oracle():
    """Every vertex's interpolated custom attributes (StrokeVertex::interpolated_attributes,
    stroke.rs:2728-2746) with two attributes per point (the width factor and a second
    one): on the paths whose triangles match the oracle's, the rows are within 1e-6 of the
    oracle's (relative, at least 1) everywhere and bit for bit on at least 97% of the paths;
    the rest differ by an ulp at some flattened points, together with the positions there
    (the half width interpolates the widths the same way)."""
    n = 200
    batch, opts, widths = random_batch(n, 4)
    rng = np.random.default_rng(44)
    attrs = np.stack([widths, rng.uniform(-5, 5, len(widths)).astype(np.float32)], axis=1)
    db = DeviceBatch(batch, opts)
    b = StrokeVWBatcher(attrs, width_attribute=0, vertex_attributes=True)
    res = b.run(db, check=False)
    synchronize()
    vo, io = res.vertex_offsets, res.index_offsets
    i = res.all_indices()
    va = b.vertex_attributes.download(np.float32, 2 * res.n_vertices).reshape(-1, 2)
    matched = same_rows = 0
    for p in range(n):
        o = opts[p]
        pb, pe = int(batch.point_offsets[p]), int(batch.point_offsets[p + 1])
        rs, rv, ri, ra = O.stroke(batch.path(p), line_width=float(o["line_width"]),
                                  miter_limit=float(o["miter_limit"]),
                                  tolerance=float(o["tolerance"]),
                                  start_cap=int(o["start_cap"]), end_cap=int(o["end_cap"]),
                                  line_join=int(o["line_join"]), vertex_offset=int(vo[p]),
                                  widths=attrs[pb:pe, 0], attributes=attrs[pb:pe])
        if not np.array_equal(i[io[p]:io[p + 1]], ri):
            continue
        matched += 1
        ga = va[vo[p]:vo[p + 1]]
        assert ga.shape == ra.shape
        assert np.all(np.abs(ga - ra) <= 1e-6 * np.maximum(1.0, np.abs(ra))), p
        same_rows += np.array_equal(ga.view(np.uint32), ra.view(np.uint32))
    print(f"{matched} paths matched, {same_rows} with the same attribute rows", flush=True)
    assert matched >= 0.97 * n and same_rows >= 0.97 * matched


def forms(paths, opts, attrs=None):
    """The batch by the parallel form and by the serial kernel (one lane per path): equal
    offsets, statuses, and bytes of vertices, indices and vertex attributes.  Returns the paths
    that the first run left to the serial kernel and the windows it counted again."""
    import ctypes as C

    from lyon_amd import _lib
    from lyon_amd.batch import _Ctx
    from lyon_amd.path import PathBatch
    lib = C.CDLL(_lib.LIB_PATH)
    ctx = C.c_void_p(_Ctx.get())
    batch = paths if isinstance(paths, PathBatch) else PathBatch.from_paths(paths)
    if attrs is None:
        attrs = np.concatenate([p.attributes for p in paths])
    db = DeviceBatch(batch, opts)
    outs, serial, again = [], C.c_uint32(0), C.c_uint32(0)
    for enabled in (0, 1):
        b = StrokeVWBatcher(attrs, vertex_attributes=True)
        lib.lyg_ctx_set_vw_serial(ctx, enabled)
        try:
            res = b.run(db, vertex_offset=5)
        finally:
            lib.lyg_ctx_set_vw_serial(ctx, 0)
        if not enabled:
            lib.lyg_ctx_last_vw(ctx, C.byref(serial), C.byref(again))
        synchronize()
        rows = b.vertex_attributes.download(np.uint32, b.n_attributes * res.n_vertices)
        outs.append((res.status.copy(), res.vertex_offsets.copy(), res.index_offsets.copy(),
                     res.all_vertices().view(np.uint32).copy(), res.all_indices().copy(), rows))
    for a, b, what in zip(*outs, ("statuses", "vertex offsets", "index offsets", "vertices",
                                  "indices", "vertex attributes")):
        assert a.shape == b.shape, what
        if not np.array_equal(a, b):
            at = int(np.nonzero((a != b).reshape(len(a), -1).any(1))[0][0])
            raise AssertionError((what, at))
    assert not outs[0][0].any()
    return serial.value, again.value


@pytest.mark.parametrize("limit", [0, 2 << 20, 5 << 20])
def test_without_memory_for_the_parallel_form(limit):
    """Where one of the parallel form's buffers cannot be allocated (4.4 MB per-path counts, 6.4
    MB of points) the serial kernel takes the batch."""
    import ctypes as C
    import threading

    from lyon_amd import _lib
    from lyon_amd.batch import _Ctx
    from lyon_amd.path import PathBatch
    n = 100000
    rng = np.random.default_rng(3)
    pts = rng.uniform(0, 50, (4 * n, 2)).astype(np.float32)
    batch = PathBatch(np.tile(np.array([3, 0, 0, 0, 5], np.uint8), n), pts,
                      np.arange(n + 1, dtype=np.uint32) * 5, np.arange(n + 1, dtype=np.uint32) * 4)
    widths = rng.uniform(0.5, 1.5, 4 * n).astype(np.float32)
    opts = vw_options(n, rng, 1.0, 0.1)
    opts["line_join"] = int(LineJoin.Miter)
    db = DeviceBatch(batch, opts)
    ref = StrokeVWBatcher(widths).run(db)
    want = ref.all_vertices().view(np.uint32).copy(), ref.all_indices().copy()
    lib = C.CDLL(_lib.LIB_PATH)
    lib.lyg_ctx_set_alloc_limit.argtypes = [C.c_void_p, C.c_uint64]
    lib.lyg_ctx_set_alloc_limit.restype = None
    got = []

    def fresh():  # a context of its own
        lib.lyg_ctx_set_alloc_limit(_Ctx.get(), limit)
        r = StrokeVWBatcher(widths).run(db)
        n_serial, again = C.c_uint32(0), C.c_uint32(0)
        lib.lyg_ctx_last_vw(C.c_void_p(_Ctx.get()), C.byref(n_serial), C.byref(again))
        got.append((n_serial.value, r.all_vertices().view(np.uint32).copy(),
                    r.all_indices().copy()))

    t = threading.Thread(target=fresh)
    t.start()
    t.join()
    assert got and got[0][0] == (n if limit else 0)
    assert np.array_equal(got[0][1], want[0]) and np.array_equal(got[0][2], want[1])


def vw_options(n, rng, width, tol):
    o = workloads.stroke_options(n, tolerance=tol, seed=int(rng.integers(1 << 30)))
    o["line_width"] = width
    o["line_join"] = rng.choice([0, 2, 3], n)  # no MiterClip: those paths are always serial
    o["start_cap"] = o["end_cap"] = rng.integers(0, 3, n)
    return o


@pytest.mark.parametrize("seed", [5, 6])
def test_the_two_forms_agree(seed):
    n = 400
    batch, opts, widths = random_batch(n, seed)
    attrs = np.stack([widths, np.arange(len(widths), dtype=np.float32)], axis=1)
    serial, _ = forms(batch, opts, attrs)
    assert serial < n


@pytest.mark.parametrize("points,all_serial", [((1, 2, 3, 4, 5), True), ((2, 5, 6), False),
                                               ((6, 7), False)])
@pytest.mark.parametrize("join", [LineJoin.Miter, LineJoin.MiterClip])
def test_short_paths_around_where_the_parallel_form_starts(points, all_serial, join):
    """Batches of a few paths of at most five points, or of clipped miters alone, are walked by
    the serial kernel; one path of six points brings the parallel form.  Plain calls of the same
    paths match the oracle."""
    rng = np.random.default_rng(len(points))
    paths = []
    for k in points * 4:
        b = PathBuilder(1)
        pts = rng.uniform(0, 50, (k, 2)).round(1)
        b.begin(tuple(pts[0]), [rng.uniform(0.5, 2)])
        for q in pts[1:]:
            b.line_to(tuple(q), [rng.uniform(0.5, 2)])
        b.end(len(paths) % 2 == 0)
        paths.append(b.build())
    o = vw_options(len(paths), rng, 1.0, 0.1)
    o["line_join"] = int(join)
    serial, _ = forms(paths, o)
    assert serial == (len(paths) if all_serial or join == LineJoin.MiterClip else 0)
    for path in paths:
        opts = StrokeOptions(line_width=1.0, line_join=join, start_cap=LineCap.Round,
                             end_cap=LineCap.Square, tolerance=0.1, variable_line_width=0)
        v, i = gpu_vw(path, opts)
        rv, ri = ref_vw(path, opts)
        assert np.array_equal(i, ri) and close_enough(v, rv, 50.0)


def turns(rng, at, heading, lengths, most):
    """Points one after the other from `at`, each at a turn of up to `most`; the last heading."""
    out = []
    for length in lengths:
        heading += rng.uniform(-most, most)
        at = at + length * np.array([np.cos(heading), np.sin(heading)])
        out.append(at)
    return out, heading


@pytest.mark.parametrize("lead", [0, 1, 55, 56, 57, 58, 59, 60, 61, 62])
def test_skipped_joins_around_the_window_size(lead):
    """Where a curve's width falls faster than it advances, its first join folds back and is
    skipped, and what up to four points after it emit may change with it, past the curve's end
    too: of these random curves of three points, about 1 in 300 changes the triangles of the edge
    after it.  Behind `lead` points of lines, so that the skip and what it reaches lie on both
    sides of the 63rd join."""
    rng = np.random.default_rng(40 + lead)
    paths, tol = [], []
    for _ in range(2500):
        b = PathBuilder(1)
        b.begin((0.0, 0.0), [1.0])
        at, heading = np.zeros(2), 0.0
        for _ in range(lead):
            at = at + rng.uniform((1, -2), (3, 2))
            b.line_to(tuple(at), [rng.uniform(0.5, 1)])
        at = at + rng.uniform((5, -9), (20, 9))
        steps = 10 ** rng.uniform(-0.5, 0.5, 3)
        (x, y, e), heading = turns(rng, at, rng.uniform(-np.pi, np.pi), steps, 1.2)
        w = 10 ** rng.uniform(-0.3, 1.3)
        b.line_to(tuple(at), [w])
        c1 = (-5 * at + 18 * x - 9 * y + 2 * e) / 6  # through x and y at t = 1/3 and 2/3
        c2 = (2 * at - 9 * x + 18 * y - 5 * e) / 6
        w = max(0.05, w - 3 * steps[0] * rng.uniform(0.3, 1))
        b.cubic_bezier_to(tuple(c1), tuple(c2), tuple(e), [w])
        for q in turns(rng, e, heading, 10 ** rng.uniform(-0.7, 1, 4), np.pi)[0]:
            b.line_to(tuple(q), [w * rng.uniform(0.2, 2)])
        b.end(False)
        paths.append(b.build())
        second = max(np.hypot(*(at - 2 * c1 + c2)), np.hypot(*(c1 - 2 * c2 + e)))
        tol.append(6 * second / (8 * 6.25))  # Wang: n = sqrt(6 second / (8 tol)) = 2.5, so 3
    opts = vw_options(len(paths), rng, 2.0, 0.1)
    opts["tolerance"] = tol
    opts["line_join"][::2] = int(LineJoin.Miter)
    serial, again = forms(paths, opts)
    print(f"{serial} of {len(paths)} paths serial, {again} windows counted again", flush=True)
    assert again > len(paths) // 10 and serial < len(paths) // 10


@pytest.mark.parametrize("closed", [False, True])
def test_many_skipped_joins_in_a_row(closed):
    """Curves of a few to hundreds of points whose first joins are skipped, one or dozens in a
    row, across window borders and up to the curve's end."""
    rng = np.random.default_rng(60 + closed)
    paths = []
    for lead in list(range(67)) * 3:
        b = PathBuilder(1)
        at = np.zeros(2)
        b.begin(tuple(at), [1.0])
        for _ in range(lead):
            at = at + rng.uniform((1, -3), (4, 3))
            b.line_to(tuple(at), [rng.uniform(0.5, 1)])
        for _ in range(int(rng.integers(1, 5))):
            size = 10 ** rng.uniform(0.3, 2)
            at = at + rng.uniform(2, 30, 2)
            b.line_to(tuple(at), [rng.uniform(0.5, 2) * size])
            q = [tuple(at + rng.uniform(-size, size, 2)) for _ in range(2)]
            at = at + rng.uniform(-size, size, 2)
            if rng.random() < 0.3:
                b.quadratic_bezier_to(q[0], tuple(at), [rng.uniform(0.01, 2)])
            else:
                b.cubic_bezier_to(*q, tuple(at), [rng.uniform(0.01, 2)])
            for _ in range(int(rng.integers(0, 3))):
                at = at + rng.uniform(-3, 3, 2)
                b.line_to(tuple(at), [rng.uniform(0.2, 2)])
        b.end(closed)
        paths.append(b.build())
    serial, again = forms(paths, vw_options(len(paths), rng, 2.0, 0.02))
    print(f"{serial} of {len(paths)} paths serial, {again} windows counted again", flush=True)
    assert again > len(paths) and serial < len(paths) // 2


def test_more_skipped_joins_than_windows():
    """Short paths whose every curve starts with a skipped join: more of them than windows, and
    none of the paths is left to the serial kernel."""
    rng = np.random.default_rng(70)
    paths = []
    for _ in range(2000):
        b = PathBuilder(1)
        at = rng.uniform(0, 100, 2)
        b.begin(tuple(at), [8.0])
        for _ in range(6):
            b.cubic_bezier_to(*[tuple(at + (3.0 * k, 0.4 * (k % 3))) for k in (1, 2, 3)], [2.0])
            at = at + (9.0, 3.0)
            b.line_to(tuple(at), [8.0])
        b.end(False)
        paths.append(b.build())
    serial, again = forms(paths, vw_options(len(paths), rng, 2.0, 0.02))
    assert serial == 0 and again >= len(paths)


def test_skips_where_rounding_makes_them():
    """Far from the origin the points of a curve lie on a coarse grid and any of its joins may
    seem to fold back, in groups close together: whichever thread settles them, the bytes are
    the serial kernel's."""
    rng = np.random.default_rng(50)
    paths = []
    for k in range(300):
        far = 10 ** rng.uniform(4, 6.5)
        b = PathBuilder(1)
        b.begin((far, far), [rng.uniform(1, 50)])
        for _ in range(6):
            q = [tuple(far + rng.uniform(0, 40, 2)) for _ in range(3)]
            b.cubic_bezier_to(*q, [rng.uniform(0.1, 50)])
        b.end(k % 2 == 0)
        paths.append(b.build())
    for tol in (0.1, 1e-3):
        serial, again = forms(paths, vw_options(len(paths), rng, 2.0, tol))
        print(f"{serial} of {len(paths)} paths serial, {again} windows again", flush=True)
        assert again > 0
