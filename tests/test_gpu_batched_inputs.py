"""What the batched call takes as a path, with the dense kernels on and off, for
paths that they hold and paths that they hand on: its own range of the input by
the offsets, wherever in the arrays that lies; verbs that consume exactly its
points; weights for each of its conics, and more than those ignored."""
import dataclasses

import numpy as np
import pytest

import oracle_ref
from ochre_amd import _lib
from ochre_amd import workloads as W
from parity import compare

pytestmark = pytest.mark.gpu

MODES = ["batched", "dense"]


def _large(seed):
    """A path of about 20 x 20 tiles: over every dense instance."""
    return W.glyph_run(1, seed=seed, smin=158.0, smax=160.0)


def _conics(seed, n=3):
    """A contour of n conics; one weight each."""
    p = np.random.default_rng(seed).uniform(2.0, 30.0, (2 * n + 1, 2)).astype(np.float32)
    return [W.MOVE] + [W.CONIC] * n + [W.CLOSE], p, np.linspace(0.5, 2.0, n).astype(np.float32)


def _with_extra(b, k, points=0, weights=0):
    """The batch with points or weights left over at the end of path k."""
    po, wo = b.point_off.copy(), b.weight_off.copy()
    pts = np.insert(b.points, [po[k + 1]] * points, [[5.0, 6.0]] * points, axis=0) if points else b.points
    w = np.insert(b.weights, [wo[k + 1]] * weights, [1.25] * weights).astype(np.float32) if weights else b.weights
    po[k + 1:] += points
    wo[k + 1:] += weights
    return dataclasses.replace(b, points=pts.astype(np.float32), point_off=po, weights=w, weight_off=wo)


def _status(ctx, b, mode):
    from ochre_amd.device import run_to_host
    with pytest.raises(_lib.OchreError) as e:
        run_to_host(ctx, b, mode, 4096, 4096)
    return e.value.status


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("first,last", [(0, 9), (1, 9), (4, 9), (4, 6), (8, 9)])
def test_a_range_of_a_batch(gpu_ctx, first, last, mode):
    """Offsets that start at a later path of the arrays, as a program that draws a part of
    a document passes them."""
    from ochre_amd.device import DeviceOutput, dense_params, rasterize_batched, set_dense_params, upload
    import torch
    b = W.concat([W.glyph_run(3, seed=5), W.from_paths([_conics(1), _conics(2)], W.IDENTITY), _large(6),
                  W.glyph_run(2, seed=7), W.from_paths([_conics(3)], W.IDENTITY)])
    db = upload(b)
    part = dataclasses.replace(db, n_paths=last - first, verb_off=db.verb_off[first:last + 1],
                               point_off=db.point_off[first:last + 1], weight_off=db.weight_off[first:last + 1],
                               xforms=db.xforms[6 * first:6 * last], n_verbs=int(b.verb_off[last]),
                               n_points=int(b.point_off[last]), n_weights=int(b.weight_off[last]))
    ref = oracle_ref.run_batch(b.subset(range(first, last)))
    out = DeviceOutput(last - first, 4096, 4096)
    was = dense_params(gpu_ctx)
    set_dense_params(gpu_ctx, mode == "dense", was["dense_groups_per_cu"], was["dense_waves_per_group"])
    try:
        rasterize_batched(gpu_ctx, part, out)
        torch.cuda.synchronize()
    finally:
        set_dense_params(gpu_ctx, bool(was["dense"]), was["dense_groups_per_cu"], was["dense_waves_per_group"])
    compare(ref, out.to_host(), max_lsb=1 if mode == "dense" else 0)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("k", [0, 3, 6])
def test_weights_left_over_are_ignored(gpu_ctx, k, mode):
    from ochre_amd.device import run_to_host
    b = W.concat([W.from_paths([_conics(11)], W.IDENTITY), W.glyph_run(2, seed=12), W.from_paths([_conics(13, 5)], W.IDENTITY),
                  W.glyph_run(2, seed=14), W.from_paths([_conics(15)], W.IDENTITY)])
    compare(oracle_ref.run_batch(b), run_to_host(gpu_ctx, _with_extra(b, k, weights=2), mode),
            max_lsb=1 if mode == "dense" else 0)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("k", [0, 3, 6])
def test_a_missing_weight_is_refused(gpu_ctx, k, mode):
    """Also where the next path's weights would follow in the array."""
    b = W.concat([W.from_paths([_conics(11)], W.IDENTITY), W.glyph_run(2, seed=12), W.from_paths([_conics(13, 5)], W.IDENTITY),
                  W.glyph_run(2, seed=14), W.from_paths([_conics(15)], W.IDENTITY)])
    wo = b.weight_off.copy()
    wo[k + 1:] -= 1
    short = dataclasses.replace(b, weights=np.delete(b.weights, wo[k + 1]), weight_off=wo)
    assert _status(gpu_ctx, short, mode) == -1


@pytest.mark.parametrize("mode", MODES + ["draw_batched", "draw_dense", "stroke_batched", "stroke_dense"])
@pytest.mark.parametrize("where", ["first", "middle", "last", "handed on", "last, handed on", "empty", "last, empty"])
def test_points_left_over_are_refused(gpu_ctx, where, mode):
    """A path, also the last one or one without verbs, that has more points than its verbs consume."""
    empty = W.from_paths([([], [])], W.IDENTITY)
    glyphs = W.glyph_run(5, seed=21)
    b, k = {"first": (glyphs, 0), "middle": (glyphs, 2), "last": (glyphs, 4),
            "handed on": (W.concat([glyphs, _large(22), W.glyph_run(3, seed=23)]), 5),
            "last, handed on": (W.concat([glyphs, _large(22)]), 5),
            "empty": (W.concat([glyphs, empty, glyphs]), 5),
            "last, empty": (W.concat([glyphs, empty]), 5)}[where]
    b = _with_extra(b, k, points=1)
    if mode.startswith(("draw", "stroke")):
        b = W.with_widths(b, 0.5, 2.0, 3)
        b.strokes = np.zeros(b.n_paths, np.uint8)  # (draw: fills, which pass through the stroke stage)
    assert _status(gpu_ctx, b, mode) == -1


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n", [1, 6])
def test_paths_without_verbs(gpu_ctx, n, mode):
    """One zero tile each (rasterizer.rs:193-198), in front of, among and after others."""
    from ochre_amd.device import run_to_host
    empty = W.from_paths([([], [])] * n, W.IDENTITY)
    b = W.concat([empty, W.glyph_run(2, seed=31), empty, W.glyph_run(1, seed=32), empty])
    compare(oracle_ref.run_batch(b), run_to_host(gpu_ctx, b, mode), max_lsb=1 if mode == "dense" else 0)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("where", ["alone", "first", "last"])
@pytest.mark.parametrize("short", [1, 400])
def test_missing_points_are_refused(gpu_ctx, where, short, mode):
    """Verbs that consume more points than the path, and the arrays, have."""
    glyphs = W.glyph_run(3, seed=41)
    p = np.random.default_rng(42).uniform(1.0, 20.0, (502 - short, 2)).astype(np.float32)
    b = W.from_paths([([W.MOVE] + [W.LINE] * 501 + [W.CLOSE], p)], W.IDENTITY)
    b = {"alone": b, "first": W.concat([b, glyphs]), "last": W.concat([glyphs, b])}[where]
    assert _status(gpu_ctx, b, mode) == -1


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("limits", [(16, 64), (0, 64), (16, 0)])
def test_small_pass_limits_refuse_no_small_path(gpu_ctx, limits, mode):
    """The plain pipeline's pass limits cut a batch into ranges; a path of up to 8,192 lines
    within 32 x 32 tiles is rasterised by the batched call whatever they are."""
    from ochre_amd.device import run_to_host, set_pass_limits
    b = W.concat([W.glyph_run(4, seed=51), _large(52), W.from_paths([_conics(53)], W.IDENTITY), _large(54)])
    set_pass_limits(gpu_ctx, *limits)
    try:
        got = run_to_host(gpu_ctx, b, mode, 4096, 4096)
    finally:
        set_pass_limits(gpu_ctx, 0, 0)
    compare(oracle_ref.run_batch(b), got, max_lsb=1 if mode == "dense" else 0)


@pytest.mark.parametrize("limits", [(0, 0), (1000, 0), (0, 8000), (60, 500)])
@pytest.mark.parametrize("n", [1, 3, 40])
def test_ordered_batches_against_the_oracle(gpu_ctx, n, limits):
    """The call with the dense kernels off, in one pass and in several, and with outputs that
    only a second call finds room in: every byte the oracle's."""
    from ochre_amd.device import run_to_host, set_pass_limits
    b = W.concat([W.glyph_run(n, seed=60 + n), W.random_paths(n, 60 + n)])
    set_pass_limits(gpu_ctx, *limits)
    try:
        got = run_to_host(gpu_ctx, b, "batched", 8, 1)
    finally:
        set_pass_limits(gpu_ctx, 0, 0)
    compare(oracle_ref.run_batch(b), got, max_lsb=0)
