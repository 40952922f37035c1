"""The adjoint's input errors on paths that go to its large-path kernels before one
wave has looked them through: verbs that consume more or fewer points than the path
has, conics without a weight, an unknown verb.  Refused, and nothing is read past
the path."""
import dataclasses

import numpy as np
import pytest

from ochre_amd import _lib
from ochre_amd import workloads as W

pytestmark = pytest.mark.gpu


def _line_path(n, points):
    p = np.random.default_rng(n + points).uniform(1.0, 60.0, (points, 2)).astype(np.float32)
    return [W.MOVE] + [W.LINE] * n + [W.CLOSE], p


def _conic_path(n, weights):
    p = np.random.default_rng(n).uniform(1.0, 60.0, (2 * n + 1, 2)).astype(np.float32)
    return [W.MOVE] + [W.CONIC] * n + [W.CLOSE], p, np.ones(weights, np.float32)


def _far_cubics(n, points):
    """Curves of thousands of lines: over one wave's lines from their steps alone."""
    p = (np.random.default_rng(n).uniform(-1.0, 1.0, (points, 2)) * 6000.0).astype(np.float32)
    return [W.MOVE] + [W.CUBIC] * n + [W.CLOSE], p


PATHS = {
    "points missing": _line_path(1500, 100),
    "one point missing": _line_path(1500, 1500),
    "a point left over": _line_path(1500, 1502),
    "weights missing": _conic_path(1100, 600),
    "unknown verb": ([W.MOVE] + [W.LINE] * 700 + [9] + [W.LINE] * 700, _line_path(1400, 1401)[1]),
    "a Move past the points": ([W.MOVE] + [W.LINE] * 1100 + [W.MOVE] + [W.LINE] * 3, _line_path(1100, 1050)[1]),
    "curves' points missing": _far_cubics(200, 301),
}


@pytest.mark.parametrize("where", ["alone", "first", "last"])
@pytest.mark.parametrize("name", list(PATHS))
def test_large_paths_with_bad_input_are_refused(gpu_ctx, name, where):
    import torch
    from ochre_amd.device import DeviceOutput, coverage_adjoint, rasterize_batched, upload
    bad = W.from_paths([PATHS[name]], W.IDENTITY)
    glyphs = W.adjoint_glyphs(n=3)
    b = {"alone": bad, "first": W.concat([bad, glyphs]), "last": W.concat([glyphs, bad])}[where]
    tb = W.adjoint_glyphs(n=b.n_paths)
    target = DeviceOutput(b.n_paths, b.n_paths * 128, b.n_paths * 16, coverage=True)
    rasterize_batched(gpu_ctx, upload(tb), target)
    print(f"[adjoint input] {name}, {where}", flush=True)
    with pytest.raises(_lib.OchreError) as e:
        coverage_adjoint(gpu_ctx, upload(b), target)
    assert e.value.status == -1
    torch.cuda.synchronize()
