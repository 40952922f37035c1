"""How large an increment's area and height get where the unordered tile stage
converts them through 32 bits (units of 2^-30: magnitudes below 2): the DDA's own
f32 steps over near-diagonal lines of the greatest length that is converted so, where
the accumulated crossing parameters drift furthest from the pixels, and over longer
ones, which need the 64-bit conversion."""
import os
import re

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
f32 = np.float32


def narrow_px():
    """The length, on its longer axis, of the longest line that converts through 32 bits."""
    src = open(os.path.join(ROOT, "ochre_amd", "csrc", "raster_common.hpp")).read()
    return int(re.search(r"FX_NARROW_PX = (\d+)\.0f", src).group(1))


def largest_increment(a, b):
    """max |area|, max |height| over the increments of the lines a -> b (rasterizer.rs:72-116)."""
    a, b = a.astype(f32), b.astype(f32)
    d = b - a
    inv = f32(1.0) / d
    step = np.abs(inv)
    sign = np.where(d < 0, -1, 1)
    xy = np.floor(a).astype(np.int64)
    edge = np.where(d > 0, xy + 1, xy).astype(f32)
    nxt = np.minimum(inv * (edge - a), f32(1.0))
    p0 = a.copy()
    area_max = height_max = 0.0
    while len(a):
        by_y = nxt[:, 1] < nxt[:, 0]
        t = np.where(by_y, nxt[:, 1], nxt[:, 0])[:, None]
        p1 = (f32(1.0) - t) * a + t * b
        h = p1[:, 1] - p0[:, 1]
        right = (xy[:, 0] + 1).astype(f32)
        area = f32(0.5) * h * ((right - p0[:, 0]) + (right - p1[:, 0]))
        area_max = max(area_max, float(np.abs(area).max()))
        height_max = max(height_max, float(np.abs(h).max()))
        moved = np.stack([~by_y, by_y], 1)
        nxt = np.where(moved, np.minimum(nxt + step, f32(1.0)), nxt)
        on = t[:, 0] != 1.0
        xy = (xy + moved * sign)[on]
        p0 = p1[on]
        a, b, nxt, step, sign = a[on], b[on], nxt[on], step[on], sign[on]
    return area_max, height_max


def lines(span, n, seed):
    """n lines of about `span` px on their longer axis, near the diagonal, anywhere within +-30000."""
    rng = np.random.default_rng(seed)
    dx = span * rng.uniform(0.97, 1.0, n)
    dy = dx * np.where(rng.random(n) < 0.7, 1.0 + rng.normal(0.0, 2e-3, n), rng.uniform(0.5, 1.0, n))
    d = np.stack([dx, np.minimum(dy, span)], 1) * rng.choice([-1.0, 1.0], (n, 2))
    lo, hi = np.maximum(-d, 0.0) - 30000.0, 30000.0 - np.maximum(d, 0.0)
    a = lo + rng.random((n, 2)) * (hi - lo)
    return a, a + d


@pytest.mark.parametrize("seed", range(4))
def test_increments_of_shorter_lines_fit_32_bits(seed):
    area, height = largest_increment(*lines(narrow_px(), 200, seed))
    # 1 + the drift's bound, span^2 * 2^-25 px, plus the rounding of coordinates of up to 30000
    assert height < 1.02 and area < 1.02 * (1.0 + 0.52)
    assert int(2.0 ** 30 * area) < 2 ** 31


def test_longer_lines_do_not():
    """Why the length decides: these increments do not fit."""
    area, height = largest_increment(*lines(30000.0, 20, 7))
    assert area > 2.0 and height < 1.1
