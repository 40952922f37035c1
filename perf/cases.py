"""The work that programs have this framework do, as cases that can be timed.

A case names a family, one of the public ways in, and its sizes:

  fill     one path through the drop-in Rasterizer: fill or stroke, finish,
           TileBuilder calls.  What a program that draws shape by shape does.
  plain    rasterize_plain over a batch on the device: bit-exact sums, paths in
           order.
  batched  rasterize_batched with its defaults (the dense kernels in front), with
           the f32 coverage that a compositor or an adjoint's target reads.  Paths
           come in the order they finish, so a pass ends with the gather that puts
           them in path order.
  stroke   ochre_stroke_batched with the same options.
  draw     a draw list of fills and strokes (an SVG's) through the ordered
           kernels, then the atlas, vertices and indices of the demo's Builder.
  adjoint  loss and gradients of the coverage against a rendered target: one step
           of fitting paths to an image.

Shapes: `glyphs` (text: 12-48 px, a few contours), `blobs` (one self-intersecting
contour of many cubics, as in illustrations and maps), `scene` (19 glyphs, turned
and scaled, to each blob).  Sizes follow the repository's own workloads.

exact() evaluates the same curves and clip points in 64 bits; the decisions that
fix which tiles exist (how many lines a curve flattens to, which pixels a line
visits) are the 32-bit ones that the reference defines, restated here.
"""
import math

import numpy as np
import torch

import ochre_amd
from ochre_amd import workloads as W
from ochre_amd.device import (Context, DeviceOutput, build_atlas, coverage_adjoint, draw as draw_list, rasterize_batched,
                              rasterize_plain, set_dense_params, stroke, upload)

_contexts = {}


def listed():
    return [
        # the smallest call: one glyph filled through the Rasterizer, latency alone
        {"name": "fill_one_glyph", "family": "fill", "stroke": False, "px": 36.0},
        # a line of text, bit-exact: a handful of paths, launches and synchronisations count
        {"name": "plain_text_line", "family": "plain", "shape": "glyphs", "n": 61},
        # a line of text with the defaults, as a serving loop that gets new text on each call sends it
        {"name": "batched_text_line", "family": "batched", "shape": "glyphs", "n": 61},
        # the repository's headline workload: a page of text
        {"name": "plain_glyph_run", "family": "plain", "shape": "glyphs", "n": 10000},
        {"name": "batched_glyph_run", "family": "batched", "shape": "glyphs", "n": 10000},
        # large paths, far over one workgroup's grid: maps and illustrations
        {"name": "plain_blobs", "family": "plain", "shape": "blobs", "n": 24, "cubics": 20000},
        {"name": "batched_blobs", "family": "batched", "shape": "blobs", "n": 24, "cubics": 20000},
        # the mix of small and large paths that a scene holds
        {"name": "batched_scene", "family": "batched", "shape": "scene", "n": 4000, "cubics": 20000},
        # outlined text
        {"name": "stroked_glyphs", "family": "stroke", "n": 5003},
        # an SVG document's draw list into the demo's atlas
        {"name": "draw_list_atlas", "family": "draw", "n": 305, "atlas": 2048},
        # fitting small shapes to a target, all of a batch at once
        {"name": "adjoint_glyphs", "family": "adjoint", "shape": "glyphs", "n": 4096, "cubics": 16},
        # fitting one large outline: a path over one wave's limits
        {"name": "adjoint_blobs", "family": "adjoint", "shape": "blobs", "n": 2, "cubics": 1400},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    f = rng.choice(["fill", "plain", "plain", "batched", "batched", "stroke", "draw", "adjoint"])
    if f == "fill":
        return {"family": f, "stroke": rng.random() < 0.3, "px": round(rng.uniform(12.0, 96.0), 2)}
    if f in ("plain", "batched"):
        shape = rng.choice(["glyphs", "glyphs", "blobs", "scene"])
        if shape == "glyphs":
            return {"family": f, "shape": shape, "n": _log_int(rng, 3, 10000)}
        if shape == "blobs":
            return {"family": f, "shape": shape, "n": _log_int(rng, 1, 24), "cubics": _log_int(rng, 2000, 20000)}
        return {"family": f, "shape": shape, "n": _log_int(rng, 20, 2000 if f == "plain" else 4000),
                "cubics": _log_int(rng, 2000, 20000)}
    if f == "stroke":
        return {"family": f, "n": _log_int(rng, 3, 5003)}
    if f == "draw":
        return {"family": f, "n": _log_int(rng, 20, 500), "atlas": 2048}
    if rng.random() < 0.7:
        return {"family": f, "shape": "glyphs", "n": _log_int(rng, 16, 4096), "cubics": rng.randint(5, 16)}
    return {"family": f, "shape": "blobs", "n": rng.randint(1, 2), "cubics": _log_int(rng, 1100, 1400)}


# ------------------------------------------------------------------- inputs

def _turned(batch, seed, canvas):
    """The batch with a random rotation, scale (0.5-4) and place for each path."""
    rng = np.random.default_rng(seed)
    n = batch.n_paths
    th, sc = rng.uniform(0.0, 2.0 * math.pi, n), rng.uniform(0.5, 4.0, n) * batch.xforms[:, 0]
    c, s = np.cos(th) * sc, np.sin(th) * sc
    batch.xforms = np.stack([c, -s, s, c, rng.uniform(0, canvas, n), rng.uniform(0, canvas, n)], 1).astype(np.float32)
    return batch


def _batch(case, seed):
    seed = seed % (1 << 31) + 100
    f = case["family"]
    if f == "fill":
        b = W.stroked_glyphs(1, seed, canvas=512.0, smin=case["px"], smax=case["px"])
    elif f == "stroke":
        b = W.stroked_glyphs(case["n"], seed)
    elif f == "draw":
        b = W.stroked_glyphs(case["n"], seed, canvas=900.0, smin=12.0, smax=120.0)
        b.strokes = (np.random.default_rng(seed).random(b.n_paths) < 0.25).astype(np.uint8)
    elif f == "adjoint":
        b = (W.adjoint_glyphs(case["n"], seed, n_cubics=case["cubics"]) if case["shape"] == "glyphs" else
             W.star_blobs(case["n"], seed, nmin=case["cubics"], nmax=case["cubics"], rmin=120.0, rmax=250.0))
    elif case["shape"] == "glyphs":
        b = W.glyph_run(case["n"], seed)
    elif case["shape"] == "blobs":
        b = W.star_blobs(case["n"], seed, nmin=1e3, nmax=case["cubics"])
    else:
        nb = max(1, case["n"] // 20)
        b = W.concat([_turned(W.glyph_run(case["n"] - nb, seed), seed, 2048.0),
                      W.star_blobs(nb, seed, canvas=2048.0, nmin=1e3, nmax=case["cubics"], rmin=100.0, rmax=1000.0)])
    return b


def _target_batch(case, seed):
    """The adjoint's target: control points moved by N(0, 0.5 px)."""
    b = _batch(case, seed)
    s = np.repeat(b.xforms[:, 0], np.diff(b.point_off))[:, None]
    z = np.random.default_rng(seed + 7).normal(0.0, 0.5, b.points.shape)
    b.points = (b.points + (z / s)).astype(np.float32)
    return b


def _context(dense):
    """One context for the program, and one for its bit-exact work."""
    if dense not in _contexts:
        _contexts[dense] = Context(0)
        set_dense_params(_contexts[dense], enabled=dense)
    return _contexts[dense]


def _capacity(case):
    """Tiles that the outputs are given room for, whatever the seed: the mean
    over paths with a margin, or every path at its largest where they are few."""
    f, n = case["family"], case["n"]

    def room(n, mean, most):
        return int(min(n * most, 1.4 * n * mean + 3.0 * most * math.sqrt(n))) + 64

    if f == "draw":
        return room(n, 90.0, 324.0)
    if f == "adjoint":
        return n * (128 if case["shape"] == "glyphs" else 8192)
    if f == "stroke" or case["shape"] == "glyphs":
        return room(n, 22.0, 81.0)
    if case["shape"] == "blobs":
        return room(n, 0.06 * 1.48e6, 0.09 * 4e6)
    nb = max(1, n // 20)
    return room(nb, 0.06 * 3.7e5, 0.09 * 1e6) + room(n - nb, 100.0, 740.0)


def _outputs(case, n_paths, coverage):
    """Outputs with room to spare, what a pass does not write staying 0."""
    cap = _capacity(case)
    out = DeviceOutput(n_paths, cap, cap, coverage=coverage)
    for t in (out.tile_xy, out.tile_alpha, out.span_xy, out.span_w, out.tile_cov):
        if t is not None:
            t.zero_()
    return out


def prepare(case, seed):
    f = case["family"]
    b = _batch(case, seed)
    if f == "fill":
        v, p, w, xf = b.path(0)
        return {"case": case, "verbs": v, "points": p, "weights": w, "xform": xf, "width": 1.5}
    s = {"case": case, "ctx": _context(f != "draw"), "db": upload(b)}
    if f == "adjoint":
        s["target"] = _outputs(case, b.n_paths, True)
        rasterize_batched(s["ctx"], upload(_target_batch(case, seed)), s["target"])
        return s
    s["out"] = _outputs(case, b.n_paths, f in ("batched", "stroke"))
    if b.widths is not None:
        s["widths"] = torch.from_numpy(b.widths).cuda()
    if f == "draw":
        s["strokes"] = torch.from_numpy(b.strokes).cuda()
        s["colors"] = torch.from_numpy(np.random.default_rng(seed).integers(0, 256, (b.n_paths, 4), np.uint8)).cuda()
        calls = 2 * s["out"].tile_capacity
        s["vertices"] = torch.zeros((4 * calls, 12), dtype=torch.uint8, device="cuda")
        s["indices"] = torch.zeros((6 * calls,), dtype=torch.int32, device="cuda")
    elif f != "plain":
        s["ordered"] = {k: torch.zeros_like(getattr(s["out"], k)) for k in ("tile_xy", "tile_cov", "span_xy", "span_w")}
    return s


# -------------------------------------------------------------------- a pass

def _call(s, out):
    f = s["case"]["family"]
    if f == "plain":
        rasterize_plain(s["ctx"], s["db"], out)
    elif f == "batched":
        rasterize_batched(s["ctx"], s["db"], out)
    elif f == "stroke":
        stroke(s["ctx"], s["db"], s["widths"], out)
    else:
        draw_list(s["ctx"], s["db"], s["strokes"], s["widths"], out)


class _Collect(ochre_amd.TileBuilder):
    def __init__(self):
        self.at, self.alpha, self.spans = [], [], []

    def tile(self, x, y, data):
        self.at.append((x, y))
        self.alpha.append(data)

    def span(self, x, y, width):
        self.spans.append((x, y, width))


def _order(start, count, total):
    """Where the items of path 0, 1, ... lie, given each path's range."""
    count = count.to(torch.int64)
    shift = start - (torch.cumsum(count, 0) - count)
    return torch.repeat_interleave(shift, count, output_size=total) + torch.arange(total, device=shift.device)


def _in_path_order(out, to):
    t = _order(out.path_tile_start[:out.n_paths], out.path_tile_count[:out.n_paths], out.n_tiles)
    q = _order(out.path_span_start[:out.n_paths], out.path_span_count[:out.n_paths], out.n_spans)
    for k, at in (("tile_xy", t), ("tile_cov", t), ("span_xy", q), ("span_w", q)):
        torch.index_select(getattr(out, k), 0, at, out=to[k][:at.numel()])
    return {"tiles": out.path_tile_count[:out.n_paths], "spans": out.path_span_count[:out.n_paths], **to}


def run(s):
    f = s["case"]["family"]
    if f == "fill":
        r, c = ochre_amd.Rasterizer(), _Collect()
        if s["case"]["stroke"]:
            r.stroke_arrays(s["verbs"], s["points"], s["width"], s["weights"], s["xform"])
        else:
            r.fill_arrays(s["verbs"], s["points"], s["weights"], s["xform"])
        r.finish(c)
        room = (int(s["case"]["px"]) // 8 + 4) ** 2
        xy, alpha, spans = np.zeros((room, 2), np.int16), np.zeros((room, 64), np.uint8), np.zeros((room, 3), np.int32)
        xy[:len(c.at)], alpha[:len(c.at)] = c.at, c.alpha
        if c.spans:
            spans[:len(c.spans)] = c.spans
        return {"tile_xy": xy, "alpha": alpha, "spans": spans}
    if f == "adjoint":
        loss, dp, dx = coverage_adjoint(s["ctx"], s["db"], s["target"])
        return {"loss": loss, "d_points": dp, "d_transforms": dx}
    out = s["out"]
    _call(s, out)
    if f == "plain":
        n = out.n_paths
        return {"tile_start": out.path_tile_start[:n], "tiles": out.path_tile_count[:n],
                "span_start": out.path_span_start[:n], "spans": out.path_span_count[:n], "tile_xy": out.tile_xy,
                "alpha": out.tile_alpha, "span_xy": out.span_xy, "span_w": out.span_w}
    if f == "draw":
        atlas, vertices, indices = build_atlas(s["ctx"], out, s["colors"], s["case"]["atlas"])
        s["vertices"][:vertices.shape[0]] = vertices
        s["indices"][:indices.shape[0]] = indices
        return {"atlas": atlas, "vertices": s["vertices"], "indices": s["indices"]}
    return _in_path_order(out, s["ordered"])


# ---------------------------------------------------------------------- work

def _sizes(case):
    """Bytes of input and tiles of output of a case, on average: a glyph has 65
    commands, 110 points and about 0.75 tiles per pixel of its size; a blob's
    boundary touches about 0.05 R^2 tiles."""
    f = case["family"]

    def mean_square(a, b):
        return (b ** 3 - a ** 3) / (3.0 * (b - a))

    def blobs(n, cubics, lo, hi, nlo=1000.0):
        c = (cubics - nlo) / math.log(cubics / nlo) if cubics > nlo else nlo
        return n * c * 25.0, n * 0.05 * mean_square(lo, hi)

    if f == "fill":
        return 969.0, 2.2 * (case["px"] / 8.0 + 1.0) * (case["px"] / 8.0)
    if f == "adjoint":
        if case["shape"] == "blobs":
            return case["n"] * case["cubics"] * 25.0, case["n"] * 1900.0
        return case["n"] * (case["cubics"] * 25.0 + 34.0), case["n"] * 36.0
    if f == "draw":
        return case["n"] * 974.0, case["n"] * 66.0
    if f == "stroke":
        return case["n"] * 973.0, case["n"] * 20.0
    if case["shape"] == "glyphs":
        return case["n"] * 969.0, case["n"] * 19.5
    if case["shape"] == "blobs":
        return blobs(case["n"], case["cubics"], 200.0, 2000.0)
    nb = max(1, case["n"] // 20)
    b_in, tiles = blobs(nb, case["cubics"], 100.0, 1000.0)
    return b_in + (case["n"] - nb) * 969.0, tiles + (case["n"] - nb) * 80.0


def work(case):
    """Inputs read once and outputs written once."""
    b_in, tiles = _sizes(case)
    f = case["family"]
    if f == "adjoint":  # the target's tiles in, a gradient for each point out
        return {"bytes": 2.0 * b_in + 260.0 * tiles, "flops": 0.0}
    if f == "draw":  # atlas bytes, and 4 vertices and 6 indices for each tile
        return {"bytes": b_in + case["atlas"] ** 2 + 72.0 * tiles, "flops": 0.0}
    per_tile = 68.0 if f in ("fill", "plain") else 260.0
    return {"bytes": b_in + per_tile * tiles, "flops": 0.0}


# ------------------------------------------------------- the values in 64 bits

_STEPS = 4096  # more pixels than any line of these cases crosses


def _at(t, *p):
    """The Bezier curve of 2 or 3 control points after its start, by de Casteljau."""
    p = list(p)
    while len(p) > 1:
        p = [(1.0 - t)[:, None] * a + t[:, None] * b for a, b in zip(p, p[1:])]
    return p[0]


def _interval(p):
    """The flattening interval of a quadratic (3 points) or a cubic (4)."""
    norm = lambda v: torch.sqrt(v[:, 0] * v[:, 0] + v[:, 1] * v[:, 1])  # noqa: E731
    tol = torch.tensor(0.1, dtype=torch.float32, device=p[0].device).to(p[0].dtype)
    if len(p) == 3:
        return torch.sqrt(4.0 * tol / norm(p[0] - 2.0 * p[1] + p[2]))
    a = -1.0 * p[0] + 3.0 * p[1] - 3.0 * p[2] + p[3]
    b = 3.0 * (p[0] - 2.0 * p[1] + p[2])
    root8 = torch.sqrt(torch.tensor(8.0, dtype=p[0].dtype, device=p[0].device))
    return torch.sqrt(root8 * tol / torch.maximum(norm(b), norm(a + b)))


def _lines(batch, p32, p64):
    """Every path's lines: (path, start, end) in 32 bits and in 64."""
    dev = p32.device
    verbs = batch.verbs.astype(np.int64)
    npts = W.VERB_POINTS[verbs]
    g = np.cumsum(npts) - npts  # a command's first point; the point before it is where it starts
    cmds = np.diff(batch.verb_off)
    path = np.repeat(np.arange(batch.n_paths), cmds)
    first_cmd = np.zeros(verbs.size, bool)
    first_cmd[batch.verb_off[:-1]] = True
    move = np.maximum.accumulate(np.where(verbs == W.MOVE, g, -1))
    before = np.concatenate([[-1], move[:-1]])  # the open contour's Move
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    parts = []

    def add(who, a32, b32, a64, b64):
        parts.append((who, a32, b32, a64, b64))

    def straight(sel, a, b):
        a, b = t(a[sel]), t(b[sel])
        add(t(path[sel]), p32[a], p32[b], p64[a], p64[b])

    straight((verbs == W.MOVE) & ~first_cmd, g - 1, before)
    straight(verbs == W.LINE, g - 1, g)
    last = np.zeros(verbs.size, bool)
    last[batch.verb_off[1:] - 1] = True
    straight(last, g + npts - 1, move)
    for verb in (W.QUAD, W.CUBIC):
        sel = np.nonzero(verbs == verb)[0]
        if not sel.size:
            continue
        at = t(g[sel])
        q32 = [p32[at + k] for k in range(-1, int(W.VERB_POINTS[verb]))]
        q64 = [p64[at + k] for k in range(-1, int(W.VERB_POINTS[verb]))]
        dt32, dt64 = _interval(q32), _interval(q64)
        who = t(path[sel])
        t32, k = torch.zeros_like(dt32), 0
        a32, a64 = q32[0], q64[0]
        while who.numel():
            t32 = torch.clamp(t32 + dt32, max=1.0)
            k += 1
            done = t32 >= 1.0
            t64 = torch.where(done, torch.ones_like(dt64), torch.clamp(k * dt64, max=1.0))
            b32, b64 = _at(t32, *q32), _at(t64, *q64)
            add(who, a32, b32, a64, b64)
            on = ~done
            who, t32, dt32, dt64 = who[on], t32[on], dt32[on], dt64[on]
            q32, q64 = [x[on] for x in q32], [x[on] for x in q64]
            a32, a64 = b32[on], b64[on]
    who, a32, b32, a64, b64 = (torch.cat(x) for x in zip(*parts))
    on = (a32 != b32).any(1)
    return who[on], a32[on], b32[on], a64[on], b64[on]


def _increments(lines):
    """(path, x, y, area, height) of every pixel that a line visits."""
    who, a, b, a64, b64 = lines
    d = b - a
    step = torch.abs(1.0 / d)
    sign = torch.where(d < 0, -1, 1)
    xy = torch.floor(a).to(torch.int64)
    edge = torch.where(d > 0, xy + 1, xy)
    nxt = torch.clamp((1.0 / d) * (edge.to(torch.float32) - a), max=1.0)
    nxt = torch.where(d == 0, torch.full_like(nxt, math.inf), nxt)
    t64 = torch.zeros_like(a64[:, 0])
    got = []
    for _ in range(_STEPS):
        if not who.numel():
            break
        by_y = nxt[:, 1] < nxt[:, 0]
        c = torch.where(by_y, nxt[:, 1], nxt[:, 0])
        end = c == 1.0
        axis = by_y.to(torch.int64)[:, None]
        pick = lambda v: torch.gather(v, 1, axis)[:, 0]  # noqa: E731
        crossed = pick(torch.where(sign > 0, xy + 1, xy))
        span = torch.where(end, torch.ones_like(t64), pick(b64) - pick(a64))
        t1 = torch.where(end, torch.ones_like(t64), (crossed - pick(a64)) / span)
        p0 = a64 + t64[:, None] * (b64 - a64)
        p1 = torch.where(end[:, None], b64, a64 + t1[:, None] * (b64 - a64))
        height = p1[:, 1] - p0[:, 1]
        right = (xy[:, 0] + 1).to(torch.float64)
        got.append((who, xy[:, 0], xy[:, 1], 0.5 * height * ((right - p0[:, 0]) + (right - p1[:, 0])), height))
        on = ~end
        moved = torch.zeros_like(xy).scatter_(1, axis, 1)
        xy = (xy + moved * sign)[on]
        nxt = torch.where(moved.bool(), torch.clamp(nxt + step, max=1.0), nxt)[on]
        who, a64, b64, t64, sign, step = who[on], a64[on], b64[on], t1[on], sign[on], step[on]
    return [torch.cat(x) for x in zip(*got)]


_BIAS, _BITS = 1 << 12, 13  # tile coordinates lie within +-4096


def _tiles(incs):
    """The tiles' keys in order, and v (64 values a tile) before |v| is cut at 1,
    with the running heights that a place between tiles has."""
    who, x, y, area, height = incs
    key = (((who << _BITS) + (y >> 3) + _BIAS) << _BITS) + (x >> 3) + _BIAS
    keys, tile = torch.unique(key, return_inverse=True)
    at = tile * 64 + (y & 7) * 8 + (x & 7)
    zeros = torch.zeros(keys.numel() * 64, dtype=torch.float64, device=area.device)
    areas = zeros.index_add(0, at, area).view(-1, 8, 8)
    heights = zeros.index_add(0, at, height).view(-1, 8, 8)
    running = torch.cumsum(heights.sum(2), 0)  # over all tiles; less what its tile row began with
    rows, n = torch.unique_consecutive(keys >> _BITS, return_counts=True)
    start = torch.repeat_interleave(torch.cumsum(n, 0) - n, n)
    began = running[start] - heights.sum(2)[start]
    carry = running - heights.sum(2) - began
    v = carry[:, :, None] + torch.cumsum(heights, 2) - heights + areas
    return keys, v.reshape(-1, 64), (running - began)[:, 0]


def _between(keys, running, asked):
    """Coverage, 0 or 1, of places (keys) where there is no tile."""
    i = torch.searchsorted(keys, asked) - 1
    ok = (i >= 0) & ((keys[i.clamp(min=0)] >> _BITS) == (asked >> _BITS))
    return torch.where(ok & (running.detach()[i.clamp(min=0)].abs() > 0.5), 1.0, 0.0).to(torch.float64)


def _to_pixels(batch, points, xf, dtype):
    """World points of every path, by its transform, operation by operation."""
    who = torch.from_numpy(np.repeat(np.arange(batch.n_paths), np.diff(batch.point_off))).to(points.device)
    m, p = xf.to(dtype)[who], points.to(dtype)
    return torch.stack([m[:, 0] * p[:, 0] + m[:, 1] * p[:, 1] + m[:, 4],
                        m[:, 2] * p[:, 0] + m[:, 3] * p[:, 1] + m[:, 5]], 1)


def _render(batch, points=None, xf=None, origin=None):
    dev = "cuda"
    p = torch.from_numpy(batch.points).to(dev)
    x = torch.from_numpy(batch.xforms).to(dev)
    shift = torch.zeros(batch.n_paths, 6, dtype=torch.float64, device=dev)
    if origin is not None:
        shift[:, 4:] = 8.0 * origin
    p32 = _to_pixels(batch, p, x - shift.to(torch.float32), torch.float32)
    p64 = _to_pixels(batch, p if points is None else points, (x.to(torch.float64) if xf is None else xf) - shift,
                     torch.float64)
    return _tiles(_increments(_lines(batch, p32, p64)))


def _exact_adjoint(case, seed):
    """The loss and its gradients by reverse-mode differentiation."""
    b, tb = _batch(case, seed), _target_batch(case, seed)
    first = torch.from_numpy(b.point_off[:-1].copy()).cuda()
    origin = torch.floor(_to_pixels(b, torch.from_numpy(b.points).cuda(), torch.from_numpy(b.xforms).cuda(),
                                    torch.float32)[first] * 0.125).to(torch.float64)
    points = torch.from_numpy(b.points).cuda().to(torch.float64).requires_grad_()
    xf = torch.from_numpy(b.xforms).cuda().to(torch.float64).requires_grad_()
    keys, v, running = _render(b, points, xf, origin)
    # the target in the same frame: its tiles moved by whole tiles
    with torch.no_grad():
        tkeys, tv, trunning = _render(tb, origin=origin)
        tcov = tv.abs().clamp(max=1.0)

    def at(keys, cov, running, asked):
        i = torch.searchsorted(keys, asked).clamp(max=keys.numel() - 1)
        return torch.where((keys[i] == asked)[:, None], cov[i], _between(keys, running, asked)[:, None])

    t = at(tkeys, tcov, trunning, keys)
    # the derivative is taken as 0 at the kinks of min(|v|, 1)
    free = (v.detach().abs() > 1e-11) & (v.detach().abs() < 1.0 - 1e-11)
    cov = torch.where(free, v.abs(), v.detach().abs().clamp(max=1.0))
    n = b.n_paths
    loss = torch.zeros(n, dtype=torch.float64, device="cuda").index_add(0, keys >> (2 * _BITS), ((cov - t) ** 2).sum(1))
    only = torch.ones_like(tkeys, dtype=torch.bool)
    i = torch.searchsorted(keys, tkeys).clamp(max=keys.numel() - 1)
    only = keys[i] != tkeys
    apart = ((_between(keys, running, tkeys[only])[:, None] - tcov[only]) ** 2).sum(1)
    loss = loss.index_add(0, tkeys[only] >> (2 * _BITS), apart)
    loss.sum().backward()
    return {"loss": loss.detach(), "d_points": points.grad, "d_transforms": xf.grad}


def exact(case, seed):
    """Coverage, loss and gradients in 64 bits.  None where every output is a
    whole number, for strokes (their outline's points are decided in 32 bits,
    join by join), and for batches of over 25 million lines."""
    f = case["family"]
    if f == "adjoint":
        return _exact_adjoint(case, seed)
    if f != "batched" or (case["shape"] == "scene" and case["n"] > 600):
        return None
    with torch.no_grad():
        _, v, _ = _render(_batch(case, seed))
        cov = torch.zeros((_capacity(case), 64), dtype=torch.float64, device="cuda")
        cov[:v.shape[0]] = v.abs().clamp(max=1.0)
    return {"tiles": None, "spans": None, "tile_xy": None, "tile_cov": cov, "span_xy": None, "span_w": None}
