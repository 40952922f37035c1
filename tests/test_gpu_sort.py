"""The key sort of the plain pipeline over its digit widths and block sizes: keys of
2 to 26 bits (row bits by the number of tile rows, x bits by the widest path) and
entry counts around a block of either size and the line between them; alpha bytes
equal to the oracle's (sums in emission order need a stable sort)."""
import numpy as np
import pytest

import oracle_ref
from ochre_amd import workloads as W
from parity import compare

pytestmark = pytest.mark.gpu


def _lines(n, tiles, rows, seed):
    p = np.random.default_rng(seed).random((n + 1, 2)) * [8.0 * tiles, 8.0 * rows]
    return [W.MOVE] + [W.LINE] * n + [W.CLOSE], p.astype(np.float32)


@pytest.mark.parametrize("wide,rows,paths,n", [
    (1, 1, 1, 3), (120, 1, 1, 3), (200, 1, 1, 8), (700, 1, 1, 4),  # keys of 2, 8, 9 and 11 bits
    (60, 30, 30, 12), (60, 60, 30, 12), (900, 30, 30, 12),         # 16, 17, 20 bits
    (2000, 60, 30, 40), (2000, 60, 500, 6),                        # 22, 26 bits
    (5, 1, 1, 510), (5, 1, 1, 540), (5, 1, 8, 500),                # entries around 1,024 and 4,096
    (60, 8, 180, 150), (60, 8, 240, 150),                          # and around 2^18
])
def test_sorted_keys(gpu_ctx, wide, rows, paths, n):
    from ochre_amd.device import run_to_host
    v = [_lines(2 if paths > 1 else n, wide, 1, 1)] + [_lines(n, 8, rows, 2 + k) for k in range(paths - 1)]
    b = W.from_paths(v, W.IDENTITY)
    stats = compare(oracle_ref.run_batch(b), run_to_host(gpu_ctx, b, "plain"), max_lsb=0)
    assert stats["bit_exact_fraction"] == 1.0
