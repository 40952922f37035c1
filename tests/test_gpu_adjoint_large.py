"""The large-path adjoint at the edges of its tile-row kernels: grids over one
256-tile window and over 64 tiles wide, of one row and of more rows than a pass
of the span kernel takes, several contours, each gradient element against the f64 oracle adjoint (finite differences pin that
oracle elsewhere; across lines of hundreds of pixels a step crosses kinks)."""
import numpy as np
import pytest

from ochre_amd import workloads as W
from test_gpu_adjoint import _check_adjoint_against, oracle_target, perturbed

pytestmark = pytest.mark.gpu


def _bands(w, h, contours, seed):
    """A box of nearly the whole area (spans in every row) and zigzags across it."""
    rng = np.random.default_rng(seed)
    verbs, pts = [], []
    box = np.array([[1.3, 1.6], [w - 1.4, 2.1], [w - 2.2, h - 1.7], [2.4, h - 1.2]])
    for c in range(contours):
        p = box if c == 0 else rng.random((9, 2)) * [w - 4.0, h - 4.0] + 2.0
        verbs += [W.MOVE] + [W.LINE] * (len(p) - 1) + [W.CLOSE]
        pts.append(p)
    return verbs, np.concatenate(pts).astype(np.float32)


@pytest.mark.parametrize("w,h,contours", [
    (2072.0, 21.0, 3),   # 260 tiles: over one window
    (2040.0, 14.0, 1),   # 256 tiles with the margin
    (522.0, 40.0, 4),    # over 64 tiles: two steps of a span row
    (30.0, 530.0, 2),    # tall: more rows than waves
    (310.0, 300.0, 5),
])
def test_large_adjoint_row_kernels(gpu_ctx, w, h, contours):
    b = W.from_paths([_bands(w, h, contours, int(w + h))], np.array([1, 0, 0, 1, 3.7, 5.2], np.float32))
    b.name = f"bands {w:g} x {h:g}, {contours} contours"
    tgt, hosts = oracle_target(gpu_ctx, perturbed(b, 0.5, 11))
    _check_adjoint_against(gpu_ctx, b, tgt, hosts, fd_samples=0, seed=12)
