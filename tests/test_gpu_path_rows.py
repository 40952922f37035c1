"""Per-path row tables around a wave's 64 tile rows, in the ordered and the
unordered tile stage: windings entering rows beyond the 64th, empty paths between
tall ones, and a batch that is not a multiple of a workgroup's paths."""
import numpy as np
import pytest

import oracle_ref
from ochre_amd import workloads as W
from parity import compare

pytestmark = pytest.mark.gpu


def _tall(h, seed):
    """A column of spans (24 tiles wide, winding non-zero in every row) and a zigzag down it."""
    rng = np.random.default_rng(seed)
    box = np.array([[3.2, 0.4], [195.7, 1.1], [194.1, h - 0.6], [2.6, h - 1.3]])
    zig = np.stack([rng.random(12) * 190.0, np.sort(rng.random(12)) * h], 1)
    verbs = [W.MOVE] + [W.LINE] * 3 + [W.CLOSE, W.MOVE] + [W.LINE] * 11 + [W.CLOSE]
    return verbs, np.concatenate([box, zig]).astype(np.float32)


@pytest.mark.parametrize("mode", ["plain", "batched", "dense"])
@pytest.mark.parametrize("rows", [60, 63, 64, 65, 129])
def test_tall_paths(gpu_ctx, rows, mode):
    from ochre_amd.device import run_to_host
    empty = ([], np.zeros((0, 2), np.float32))
    paths = [_tall(8.0 * rows, rows), empty, _tall(8.0 * rows - 17.0, rows + 1), _tall(30.0, 2), empty, empty,
             _tall(8.0 * rows + 9.0, rows + 2)]
    b = W.from_paths(paths, np.array([1, 0, 0, 1, 5.5, 2.25], np.float32))
    compare(oracle_ref.run_batch(b), run_to_host(gpu_ctx, b, mode), max_lsb=1 if mode == "dense" else 0)
