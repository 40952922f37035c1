"""The ordered tile stage at the edges of its 64-run blocks: rows whose runs end
just before, at and after a block, all in one tile or over many, corner-to-corner
runs of 15 increments, and crossing-only groups between them; alpha bytes equal to
the oracle's (sums in emission order)."""
import numpy as np
import pytest

import oracle_ref
from ochre_amd import workloads as W
from parity import compare

pytestmark = pytest.mark.gpu


def _zigzag(n, tiles, rows, seed):
    """n lines over `tiles` x `rows` tiles; every third joins opposite corners of a tile."""
    rng = np.random.default_rng(seed)
    p = rng.random((n + 1, 2)) * [8.0 * tiles, 8.0 * rows]
    for k in range(0, n, 3):
        t = np.floor(p[k] / 8.0) * 8.0
        p[k], p[k + 1] = t + 0.03, t + [7.98, 7.96]
    return [W.MOVE] + [W.LINE] * n + [W.CLOSE], p.astype(np.float32)


@pytest.mark.parametrize("tiles,rows", [(1, 1), (5, 1), (70, 1), (9, 6)])
@pytest.mark.parametrize("n", [1, 31, 62, 63, 64, 65, 127, 191, 400])
def test_rows_of_runs_around_a_block(gpu_ctx, n, tiles, rows):
    from ochre_amd.device import run_to_host
    paths = [_zigzag(n, tiles, rows, 100 * n + k) for k in range(3)]
    b = W.from_paths(paths, np.array([[1, 0, 0, 1, 0, 0], [1, 0, 0, 1, -13.5, 4.25], [1, 0, 0, 1, 7.0, -9.0]], np.float32))
    stats = compare(oracle_ref.run_batch(b), run_to_host(gpu_ctx, b, "plain"), max_lsb=0)
    assert stats["bit_exact_fraction"] == 1.0


@pytest.mark.parametrize("n,tiles", [(2040, 1), (2047, 1), (2048, 1), (2049, 1), (2111, 3), (6143, 1), (6145, 2), (1500, 30)])
def test_rows_of_two_waves(gpu_ctx, n, tiles):
    """Rows of 2,048 entries and more (two waves to a row) beside shorter ones."""
    from ochre_amd.device import run_to_host
    paths = [_zigzag(n, tiles, 1, n), _zigzag(90, 5, 2, 1), _zigzag(n + 64, tiles, 2, 3)]
    b = W.from_paths(paths, W.IDENTITY)
    stats = compare(oracle_ref.run_batch(b), run_to_host(gpu_ctx, b, "plain"), max_lsb=0)
    assert stats["bit_exact_fraction"] == 1.0
