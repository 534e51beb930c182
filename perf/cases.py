"""The work that users of this engine have it do, as cases that can be timed and compared.

Every case goes through the Python entry points of ``lyon_amd``: single paths over host
buffers (lyon's own calls), batches over device-resident paths, lyon_geom's flattening over
segment arrays, SVG path data ingest and the two path validators.  Sizes, coordinates and
options are those of the repository's benchmark and serving workloads (``bench.py``,
``lyon_amd/workloads.py``) and small shapes as icons and text bring them; ``draw`` gives more
cases of the same ranges.

All outputs are held to the engine's own bar: lyon's f32 arithmetic step for step, so two
correct builds give the same bytes (``tolerance`` is "exact").  The flattened points, the
areas and the parsed points also have a plain float64 form (``exact``); a stroke's or a
fill's vertices are what lyon's algorithm makes of f32 predicates and have none.

Outputs land in arrays of the program's own, made once with room for any input of the case
(the used part is followed by zeros), as a renderer keeps its vertex and index buffers.
"""
import math

import numpy as np
import torch

from lyon_amd import (BuffersBuilder, FillOptions, FillRule, FillTessellator, LineCap, LineJoin,
                      Orientation, PathBatch, StrokeOptions, StrokeTessellator, VertexBuffers)
from lyon_amd import algorithms, svg, workloads
from lyon_amd.batch import (DeviceBatch, DeviceBuffer, FillBatcher, StrokeBatcher,
                            StrokeVWBatcher, flatten_segments_device)


# ---- cases -------------------------------------------------------------------------------
def listed():
    return [
        # one path drawn by an interactive program: lyon's own call, host buffers in and out
        dict(name="stroke one path", kind="stroke_path", segs=64, extent=1024.0, closed=True,
             width=4.0, join=0, cap=0, tol=0.1),
        dict(name="fill one path", kind="fill_path", segs=64, extent=1024.0, rule=0,
             orientation=1, tol=0.1),
        # a frame's worth of short strokes (the serving workload's 4-64 segment requests)
        dict(name="stroke 64 short paths", kind="stroke_batch", paths=64, min_segs=4,
             max_segs=64, extent=4096.0, closed=False, tol=0.05),
        # the benchmark's batched stroke
        dict(name="stroke 10000 paths", kind="stroke_batch", paths=10000, min_segs=8,
             max_segs=256, extent=2048.0, closed=False, tol=0.05),
        # the same paths with a width per endpoint (pen pressure, map lines)
        dict(name="variable width 10000 paths", kind="stroke_vw", paths=10000, min_segs=8,
             max_segs=256, extent=2048.0, attributes=1, tol=0.05),
        # glyphs and icons: small closed contours with holes, non-zero
        dict(name="fill 1000 glyphs", kind="fill_glyphs", paths=1000, extent=64.0, rule=1,
             tol=0.1),
        # the benchmark's batched fill: self-intersecting stars and loops of cubics
        dict(name="fill 4096 paths", kind="fill_batch", paths=4096, tol=0.05),
        # the benchmark's single large fill (a coastline, a scan): one 1M-vertex contour
        dict(name="banded fill 1M vertices", kind="fill_walk", vertices=1 << 20, extent=8192.0,
             rule=1, tol=0.1),
        # lyon_geom: the curves of the batched stroke flattened in place
        dict(name="flatten 10000 paths", kind="flatten", paths=10000, min_segs=8, max_segs=256,
             extent=2048.0, tol=0.05),
        # loading a document: path data as editors write it
        dict(name="svg 4096 strings", kind="svg", paths=4096, min_segs=8, max_segs=64,
             extent=1024.0, decimals=3, relative=False),
        # picking: many points against the paths of a scene
        dict(name="hit test 100000 points", kind="hit_test", paths=10000, min_segs=8,
             max_segs=256, extent=2048.0, queries=100000, rule=1, tol=0.05),
        # winding direction and size of every path of a scene
        dict(name="signed areas 10000 paths", kind="areas", paths=10000, min_segs=8,
             max_segs=256, extent=2048.0, tol=0.05),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["stroke_path", "fill_path", "stroke_batch", "stroke_batch", "stroke_vw",
                       "fill_glyphs", "fill_batch", "fill_walk", "flatten", "svg", "hit_test",
                       "areas"])
    extent = round(math.exp(rng.uniform(math.log(128.0), math.log(2048.0))), 2)
    tol = rng.choice([0.05, 0.1, 0.25])
    min_segs, max_segs = rng.randint(1, 12), _log(rng, 13, 256)
    if kind == "stroke_path":
        return dict(kind=kind, segs=_log(rng, 1, 512), extent=extent,
                    closed=rng.random() < 0.5, width=round(rng.uniform(0.5, 8.0), 2),
                    join=rng.randrange(4), cap=rng.randrange(3), tol=tol)
    if kind == "fill_path":
        return dict(kind=kind, segs=_log(rng, 3, 128), extent=extent, rule=rng.randrange(2),
                    orientation=rng.randrange(2), tol=tol)
    if kind == "stroke_batch":
        return dict(kind=kind, paths=_log(rng, 1, 10000), min_segs=min_segs, max_segs=max_segs,
                    extent=extent, closed=rng.random() < 0.5, tol=tol)
    if kind == "stroke_vw":
        return dict(kind=kind, paths=_log(rng, 16, 10000), min_segs=min_segs, max_segs=max_segs,
                    extent=extent, attributes=rng.randint(1, 3), tol=tol)
    if kind == "fill_glyphs":
        return dict(kind=kind, paths=_log(rng, 16, 4096), extent=rng.choice([24.0, 64.0, 200.0]),
                    rule=rng.randrange(2), tol=rng.choice([0.02, 0.1]))
    if kind == "fill_batch":
        return dict(kind=kind, paths=_log(rng, 64, 2048), tol=tol)
    if kind == "fill_walk":
        return dict(kind=kind, vertices=_log(rng, 5000, 1 << 20),
                    extent=rng.choice([2048.0, 8192.0]), rule=rng.randrange(2), tol=tol)
    if kind == "svg":
        return dict(kind=kind, paths=_log(rng, 64, 4096), min_segs=min_segs,
                    max_segs=_log(rng, 13, 64), extent=extent, decimals=rng.randint(0, 6),
                    relative=rng.random() < 0.5)
    case = dict(kind=kind, paths=_log(rng, 100, 10000), min_segs=min_segs, max_segs=max_segs,
                extent=extent, tol=tol)
    if kind == "hit_test":
        case.update(queries=_log(rng, 1000, 100000), rule=rng.randrange(2))
    return case


# ---- inputs ------------------------------------------------------------------------------
def _strokes(case, seed):
    return workloads.stroke_batch(case["paths"], case["min_segs"], case["max_segs"],
                                  case["extent"], seed=seed, closed=bool(case.get("closed")))


def _glyphs(case, seed):
    """Closed contours of 3 to 24 lines, quadratics and cubics around a centre, half of them
    with a smaller counter inside, wound the other way."""
    rng = np.random.default_rng(seed)
    verbs, points, vo, po = [], [], [0], [0]
    e = case["extent"]
    for _ in range(case["paths"]):
        c = e * (0.5 + 2.0 * rng.random(2))
        n_points = 0
        for inner in range(1 + int(rng.random() < 0.5)):
            k = int(rng.integers(3, 25))
            r = e * (0.15 if inner else 0.5) * (0.7 + 0.3 * rng.random(k))
            a = 2.0 * np.pi * (np.arange(k) + 0.3 * rng.random(k)) / k
            if inner:
                a = -a
            on = c + np.stack([r * np.cos(a), r * np.sin(a)], 1)
            nxt = np.roll(on, -1, 0)
            kinds = rng.integers(0, 3, k)
            pts = [on[:1]]
            for j in range(k):
                for m in range(kinds[j]):  # control points near the chord
                    f = (m + 1.0) / (kinds[j] + 1.0)
                    pts.append((on[j] * (1 - f) + nxt[j] * f +
                                e * 0.05 * rng.standard_normal(2))[None])
                pts.append(nxt[j:j + 1])
            pts.append(on[:1])  # Close keeps a copy of the first point
            p = np.concatenate(pts).astype(np.float32)
            p[-2] = p[0]
            verbs.append(np.concatenate([[3], kinds, [4]]).astype(np.uint8))
            points.append(p)
            n_points += len(p)
        vo.append(sum(len(v) for v in verbs[-(1 + inner):]) + vo[-1])
        po.append(po[-1] + n_points)
    return PathBatch(np.concatenate(verbs), np.concatenate(points), np.array(vo, np.uint32),
                     np.array(po, np.uint32))


def _svg_strings(case, seed):
    """Path data of stroke paths with `decimals` decimals; also the numbers as written (f64)
    and, for relative commands, the index of the current point each is relative to."""
    batch = _strokes(case, seed)
    verbs = np.asarray(batch.verbs)
    vo, po = batch.verb_offsets.astype(np.int64), batch.point_offsets.astype(np.int64)
    pts = np.asarray(batch.points, np.float64)
    d, rel = case["decimals"], bool(case["relative"])
    npv = np.array([1, 2, 3, 1, 1, 0], np.int64)[verbs]
    first = np.cumsum(npv) - npv  # each verb's first point (all paths: Begin .. End)
    base = np.repeat(first - 1, npv)
    if rel:
        opens = np.repeat(verbs == 3, npv)
        pts = np.where(opens[:, None], pts, pts - pts[np.maximum(base, 0)])
    pts = np.round(pts, d)
    pair = "%%.%df,%%.%df" % (d, d)
    word = {3: "M" + pair}
    for v, c in ((0, "L"), (1, "Q"), (2, "C")):
        word[v] = (c.lower() if rel else c) + " ".join([pair] * (v + 1))
    word[5] = ""
    strings = []
    for i in range(case["paths"]):
        form = "".join([word[v] for v in verbs[vo[i]:vo[i + 1]].tolist()])
        strings.append(form % tuple(pts[po[i]:po[i + 1]].reshape(-1).tolist()))
    return strings, batch, pts, first


def _room(case):
    """Room for a case's output, whatever the seed: (vertices, indices) of a tessellation,
    (points, segments) of a flattening or of path data."""
    kind, n = case["kind"], case.get("paths", 1)
    spare = 1.2 + 7.0 / math.sqrt(n)
    if kind == "fill_glyphs":
        v = n * (40 + 105 * math.sqrt(case["extent"] / 64.0 * 0.1 / case["tol"]) * spare)
        return int(v), int(3.3 * v)
    if kind == "fill_batch":
        return int(n * 6300 * spare), int(n * 25200 * spare)
    if kind == "fill_walk":
        return 60 * case["vertices"], 84 * case["vertices"]
    if kind == "svg":
        segs = min(_segments(case) * spare, n * case["max_segs"]) + 1
        return int(3 * segs + n), int(segs + 2 * n)
    curve = math.sqrt(17.0 * case["extent"] / (8.0 * case["tol"])) + 1.0  # the longest cubic
    if kind in ("stroke_path", "fill_path"):
        segs = case["segs"]
        v = segs * (curve + segs if kind == "fill_path" else 2.2 * curve + 26.0) + 64
        return int(v), int(3.1 * v)
    segs = min(_segments(case) * spare, n * case["max_segs"]) + 1
    points = min(_segments(case) * _points_per_segment(case) * spare, segs * curve)
    if kind == "flatten":
        return int(points), int(segs)
    v = 2.3 * points + 26 * segs + 64 * n
    return int(v), int(3.1 * v)


def _buf(a):
    return DeviceBuffer.from_numpy(np.ascontiguousarray(a).reshape(-1))


class _Alias:
    """A device allocation of the library as torch sees it (no copy)."""

    def __init__(self, buf, typestr, size):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": (buf.nbytes // size,), "typestr": typestr,
                                         "data": (buf.ptr, False), "version": 2}


_TYPES = {"f4": 4, "i4": 4, "u1": 1}


def _zeros(nbytes):
    b = DeviceBuffer(nbytes)
    torch.as_tensor(_Alias(b, "|u1", 1), device="cuda").zero_()
    return b


def _tensor(state, buf, kind, n):
    """The first n values of a device buffer; the alias is made once per buffer."""
    seen = state.setdefault("aliases", {})
    key = (buf.ptr, buf.nbytes, kind)
    if key not in seen:
        seen[key] = torch.as_tensor(_Alias(buf, ("|" if kind == "u1" else "<") + kind,
                                           _TYPES[kind]), device="cuda")
    return seen[key][:n]


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind in ("hit_test", "areas"):
        room = None
    else:
        room = s["room"] = _room(case)
    if kind == "stroke_path":
        s["path"] = workloads.stroke_batch(1, case["segs"], case["segs"], case["extent"],
                                           seed=seed, closed=bool(case["closed"])).path(0)
        s["opts"] = StrokeOptions(line_width=case["width"], tolerance=case["tol"],
                                  line_join=LineJoin(case["join"]),
                                  start_cap=LineCap(case["cap"]), end_cap=LineCap(case["cap"]))
        s["tess"] = StrokeTessellator()
    elif kind == "fill_path":
        s["path"] = workloads.stroke_batch(1, case["segs"], case["segs"], case["extent"],
                                           seed=seed, closed=True).path(0)
        s["opts"] = FillOptions(tolerance=case["tol"], fill_rule=FillRule(case["rule"]),
                                sweep_orientation=Orientation(case["orientation"]))
        s["tess"] = FillTessellator()
    elif kind == "stroke_batch":
        s["db"] = DeviceBatch(_strokes(case, seed),
                              workloads.stroke_options(case["paths"], tolerance=case["tol"],
                                                       seed=seed))
        s["batcher"] = StrokeBatcher()
    elif kind == "stroke_vw":
        batch = _strokes(case, seed)
        rng = np.random.default_rng(seed)
        widths = rng.uniform(0.5, 2.0, (len(batch.points), case["attributes"]))
        s["db"] = DeviceBatch(batch, workloads.stroke_options(case["paths"],
                                                              tolerance=case["tol"], seed=seed))
        s["batcher"] = StrokeVWBatcher(widths.astype(np.float32), case["attributes"] - 1,
                                       vertex_attributes=case["attributes"] > 1)
        if case["attributes"] > 1:
            s["batcher"].vertex_attributes = _zeros(4 * case["attributes"] * room[0])
    elif kind in ("fill_glyphs", "fill_batch", "fill_walk"):
        n = case.get("paths", 1)
        if kind == "fill_batch":
            batch = workloads.fill_batch(n, seed=seed)
            opts = workloads.fill_options(n, tolerance=case["tol"], seed=seed)
        else:
            batch = _glyphs(case, seed) if kind == "fill_glyphs" else PathBatch.from_paths(
                [workloads.random_walk_path(case["vertices"], seed=seed, extent=case["extent"])])
            opts = workloads.one_fill_options(case["tol"], case["rule"])
        s["db"] = DeviceBatch(batch, opts)
        s["batcher"] = FillBatcher(banded=kind == "fill_walk")
    elif kind == "flatten":
        kinds, ctrl = workloads.segments_of(_strokes(case, seed))
        s["n"] = len(kinds)
        s["kinds"], s["ctrl"] = _buf(kinds), _buf(ctrl)
        s["points"], s["offsets"] = _zeros(8 * room[0]), _zeros(4 * (room[1] + 1))
    elif kind == "svg":
        text, offsets = svg.pack_strings(_svg_strings(case, seed)[0])
        s["text"], s["offsets"] = _buf(text), _buf(offsets)
        out = s["out"] = svg.DeviceSvgBatch()
        n = out.n = case["paths"]
        out.points, out.verbs = _zeros(8 * room[0]), _zeros(room[1])
        out.verb_offsets, out.point_offsets = _zeros(4 * (n + 1)), _zeros(4 * (n + 1))
        out.errors = _zeros(16 * n)
    else:
        s["db"] = DeviceBatch(_strokes(case, seed))
        if kind == "hit_test":
            rng = np.random.default_rng(seed)
            q = case["queries"]
            s["xy"] = _buf((rng.random((q, 2)) * case["extent"]).astype(np.float32))
            s["of"] = _buf(rng.integers(0, case["paths"], q).astype(np.uint32))
            s["winding"], s["inside"] = DeviceBuffer(4 * q), DeviceBuffer(q)
        else:
            s["areas"] = DeviceBuffer(4 * case["paths"])
    if kind in ("stroke_path", "fill_path"):
        s["vertices"] = np.zeros((room[0], 2), np.float32)
        s["indices"] = np.zeros(room[1], np.uint32)
    if "batcher" in s:
        s["batcher"].vertices, s["batcher"].indices = _zeros(8 * room[0]), _zeros(4 * room[1])
    torch.cuda.synchronize()
    return s


# ---- one pass ----------------------------------------------------------------------------
def run(s):
    case, kind = s["case"], s["kind"]
    if kind in ("stroke_path", "fill_path"):
        out = VertexBuffers()
        s["tess"].tessellate_path(s["path"], s["opts"], BuffersBuilder(out))
        s["vertices"][:len(out.vertices)] = out.vertices
        s["indices"][:len(out.indices)] = out.indices
        return {"vertices": s["vertices"], "indices": s["indices"].view(np.int32)}
    if "batcher" in s:
        fill = kind.startswith("fill")
        r = s["batcher"].run(s["db"], check=not fill)
        out = {"vertices": _tensor(s, r.vertices, "f4", 2 * s["room"][0]),
               "indices": _tensor(s, r.indices, "i4", s["room"][1]),
               "vertex_offsets": _tensor(s, r.voffs, "i4", r.n + 1),
               "index_offsets": _tensor(s, r.ioffs, "i4", r.n + 1)}
        if case.get("attributes", 1) > 1:
            out["attributes"] = _tensor(s, s["batcher"].vertex_attributes, "f4",
                                        case["attributes"] * s["room"][0])
        if fill:
            out["status"] = _tensor(s, r.status_buf, "i4", r.n)
        return out
    if kind == "flatten":
        flatten_segments_device(s["kinds"], s["ctrl"], s["n"], case["tol"], s["points"],
                                s["offsets"])
        return {"points": _tensor(s, s["points"], "f4", 2 * s["room"][0]),
                "offsets": _tensor(s, s["offsets"], "i4", s["room"][1] + 1)}
    if kind == "svg":
        r = s["out"] = svg.parse_paths_device(s["text"], s["offsets"], case["paths"],
                                              out=s["out"])
        return {"verbs": _tensor(s, r.verbs, "u1", s["room"][1]),
                "points": _tensor(s, r.points, "f4", 2 * s["room"][0]),
                "verb_offsets": _tensor(s, r.verb_offsets, "i4", r.n + 1),
                "point_offsets": _tensor(s, r.point_offsets, "i4", r.n + 1),
                "errors": _tensor(s, r.errors, "i4", 4 * r.n)}
    if kind == "hit_test":
        q = case["queries"]
        algorithms.winding_numbers_device(s["db"], s["xy"], s["of"], q, case["tol"],
                                          FillRule(case["rule"]), s["winding"], s["inside"])
        return {"winding": _tensor(s, s["winding"], "i4", q),
                "inside": _tensor(s, s["inside"], "u1", q)}
    algorithms.signed_areas_device(s["db"], case["tol"], s["areas"])
    return {"areas": _tensor(s, s["areas"], "f4", case["paths"])}


# ---- what a pass cannot do without -------------------------------------------------------
def _segments(case):
    lo, hi = case["min_segs"], case["max_segs"]
    return case["paths"] * (hi - lo) / math.log(hi / lo)


def _points_per_segment(case):
    """Wang counts of curves through uniform points (a quarter lines, a quarter quadratics,
    half cubics)."""
    k = case["extent"] / (8.0 * case["tol"])
    return 0.25 + 0.25 * max(1.0, math.sqrt(1.8 * k)) + 0.5 * max(1.0, math.sqrt(6.6 * k))


def work(case):
    """Bytes: inputs once, outputs once (sizes from the generators' mean counts).  Flops: the
    evaluation of each flattened point (about 12) and, where a stroke joins it to its
    neighbours, its normals and sides (about 60 more)."""
    kind = case["kind"]
    if kind == "fill_glyphs":  # 44 points in, 104 vertices, 105 triangles out
        n = case["paths"] * math.sqrt(case["extent"] / 64.0 * 0.1 / case["tol"])
        return {"bytes": n * (25 + 8 * 44 + 8 * 104 + 12 * 105), "flops": n * 104 * 60}
    if kind == "fill_batch":  # 6,200 vertices, 8,200 triangles a path
        n = case["paths"]
        return {"bytes": n * (8 * 400 + 8 * 6200 + 12 * 8200), "flops": n * 6200 * 60}
    if kind == "fill_walk":  # trapezoids: 0.44 triangles a vertex; longer walks cross more
        n = case["vertices"]
        v = n * ((11.0 if case["rule"] else 7.5) + 3.0 * math.log(n / 5000.0))
        return {"bytes": 9 * n + v * (8 + 12 * 0.44), "flops": v * 20}
    if kind in ("stroke_path", "fill_path"):
        case = dict(case, paths=1, min_segs=case["segs"], max_segs=case["segs"] + 1e-6)
    segs = _segments(case)
    inputs = segs * (1 + 8 * 2.25)
    if kind == "svg":
        digits = case["decimals"] + 4 + 0.5 * case["relative"]
        return {"bytes": segs * 2.25 * (2 * digits + 1) + segs + inputs,
                "flops": segs * 2.25 * 2 * 8}
    points = segs * _points_per_segment(case)
    if kind in ("stroke_path", "stroke_batch", "stroke_vw"):
        k = case.get("attributes", 0)
        widths = 4 * k * (segs * 2.25 + (points * 2.1 if k > 1 else 0))
        return {"bytes": inputs + widths + points * (8 * 2.1 + 4 * 6.3), "flops": points * 72}
    if kind == "fill_path":  # random curves over one box: half of all pairs of segments cross
        v = points + 0.5 * segs * segs
        return {"bytes": inputs + v * (8 + 12), "flops": v * 60}
    if kind == "flatten":
        return {"bytes": segs * 40 + points * 8, "flops": points * 12}
    if kind == "hit_test":
        per = points / case["paths"]
        return {"bytes": inputs + case["queries"] * 17, "flops": case["queries"] * per * 14}
    return {"bytes": inputs + 4 * case["paths"], "flops": points * 18}


def tolerance(case):
    return "exact"


# ---- the same in 64 bits -----------------------------------------------------------------
def _counts(kinds, ctrl, tol):
    """Flattened points of each segment and the curves' parameter step, by Wang's formula in
    f32 as lyon rounds it (the counts fix the layout of the output)."""
    f = np.float32
    c = np.asarray(ctrl, f).reshape(-1, 4, 2)
    d = f(1) / (f(8) * f(tol))
    two = f(2)
    lq = (c[:, 0] - c[:, 1] * two + c[:, 2]) * two
    v1 = (c[:, 0] - c[:, 1] * two + c[:, 2]) * f(6)
    v2 = (c[:, 1] - c[:, 2] * two + c[:, 3]) * f(6)
    sq = lambda v: v[:, 0] * v[:, 0] + v[:, 1] * v[:, 1]  # noqa: E731
    e = np.where(kinds == 1, sq(lq), np.maximum(sq(v1), sq(v2))) * d * d
    i4 = np.arange(1, 25, dtype=np.float64) ** 4
    n = np.where(e <= f(331776), np.searchsorted(i4, e.astype(np.float64)) + 1.0,
                 np.sqrt(np.sqrt(e)))
    n = np.where(kinds == 0, 1.0, n.astype(f)).astype(f)
    return n.astype(np.int64), n


def _flatten64(kinds, ctrl, tol):
    """(points f64, first point of each segment)."""
    cnt, n = _counts(kinds, ctrl, tol)
    cnt_t = torch.from_numpy(cnt)
    off = torch.cumsum(cnt_t, 0) - cnt_t
    seg = torch.repeat_interleave(torch.arange(len(cnt)), cnt_t)
    k = torch.arange(len(seg)) - off[seg] + 1
    t = k.double() / torch.from_numpy(n.astype(np.float64))[seg]
    last = k == cnt_t[seg]
    c = torch.from_numpy(np.asarray(ctrl, np.float32).reshape(-1, 4, 2)).double()
    kd = torch.from_numpy(np.asarray(kinds, np.int64))
    quad = (kd == 1)[:, None]
    a1 = torch.where(quad, 2 * (c[:, 1] - c[:, 0]), 3 * (c[:, 1] - c[:, 0]))
    a2 = torch.where(quad, c[:, 0] + c[:, 2] - 2 * c[:, 1],
                     3 * c[:, 0] - 6 * c[:, 1] + 3 * c[:, 2])
    a3 = torch.where(quad, torch.zeros_like(a1), c[:, 3] - c[:, 0] + 3 * (c[:, 1] - c[:, 2]))
    end = c[torch.arange(len(kd)), kd + 1]
    out = torch.empty((len(seg), 2), dtype=torch.float64)
    for x in range(2):
        p = ((a3[:, x][seg] * t + a2[:, x][seg]) * t + a1[:, x][seg]) * t + c[:, 0, x][seg]
        out[:, x] = torch.where(last, end[:, x][seg], p)
    return out, off


def _padded(points, room):
    out = torch.zeros((room, 2), dtype=torch.float64)
    out[:len(points)] = points
    return out.reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "flatten":
        kinds, ctrl = workloads.segments_of(_strokes(case, seed))
        return {"points": _padded(_flatten64(kinds, ctrl, case["tol"])[0], _room(case)[0]),
                "offsets": None}
    if kind == "areas":
        # open paths: Begin, segments, End; the last point joins the first
        batch = _strokes(case, seed)
        kinds, ctrl = workloads.segments_of(batch)
        p, off = _flatten64(kinds, ctrl, case["tol"])
        segs = torch.from_numpy(np.diff(batch.verb_offsets.astype(np.int64)) - 2)
        first = torch.from_numpy(batch.points.astype(np.float64))[
            torch.from_numpy(batch.point_offsets[:-1].astype(np.int64))]
        seg0 = torch.cumsum(segs, 0) - segs
        ends = torch.cat([off, torch.tensor([len(p)])])
        of = torch.repeat_interleave(torch.arange(len(segs)),
                                     ends[seg0 + segs] - ends[seg0])
        p -= first[of]
        same = torch.zeros(len(p), dtype=torch.bool)
        same[1:] = of[1:] == of[:-1]
        term = torch.zeros(len(p), dtype=torch.float64)
        term[1:] = (p[:-1, 0] * p[1:, 1] - p[:-1, 1] * p[1:, 0]) * same[1:]
        total = torch.zeros(len(segs), dtype=torch.float64)
        total.index_add_(0, of, term)
        return {"areas": 0.5 * total}
    if kind == "svg":
        _, batch, pts, first = _svg_strings(case, seed)
        if case["relative"]:
            verbs = np.asarray(batch.verbs)
            npv = np.array([1, 2, 3, 1, 1, 0], np.int64)[verbs]
            ends = first + npv - 1
            step = np.where((verbs == 5)[:, None], 0.0, pts[np.minimum(ends, len(pts) - 1)])
            at = np.cumsum(step, 0)
            for i in range(case["paths"]):  # a Begin is absolute
                v0, v1 = int(batch.verb_offsets[i]), int(batch.verb_offsets[i + 1])
                at[v0:v1] = np.cumsum(step[v0:v1], 0)
            cur = np.concatenate([np.zeros((1, 2)), at[:-1]])
            cur[verbs == 3] = 0.0
            pts = pts + np.repeat(cur, npv, 0)
        return {"verbs": None, "points": _padded(torch.from_numpy(pts), _room(case)[0]),
                "verb_offsets": None, "point_offsets": None, "errors": None}
    return None
