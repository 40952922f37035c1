"""The plain flatten's emit pass at its edges: curves of a few to several hundred
segments (t restarted from a kept value every 8 steps, 128 kept), paths of zero to
three commands (many segments per wave of the command search), lines around a
workgroup's share; outputs equal to the oracle's."""
import numpy as np
import pytest

import oracle_ref
from ochre_amd import workloads as W
from ochre_amd.device import run_to_host
from parity import compare

pytestmark = pytest.mark.gpu


def _check(ctx, paths):
    b = W.from_paths(paths, W.IDENTITY)
    compare(oracle_ref.run_batch(b), run_to_host(ctx, b, "plain"), max_lsb=0)


@pytest.mark.parametrize("segments", [1, 2, 7, 8, 9, 16, 17, 63, 64, 65, 119, 121, 127, 129, 300])
def test_curves_by_segments(gpu_ctx, segments):
    # a cubic's step is sqrt(0.1 sqrt(8) / c), c its larger second difference; a quadratic's sqrt(0.4 / c)
    c3, c2 = 0.2828 * (segments - 0.5) ** 2, 0.4 * (segments - 0.5) ** 2
    k = c3 / 6.0
    cubic = ([W.MOVE, W.CUBIC, W.CLOSE], [(10.3, 20.7), (10.3 + k, 21.0), (30.0 + k, 41.5), (31.2, 60.4)])
    quad = ([W.MOVE, W.QUAD, W.LINE, W.CLOSE], [(5.1, 9.9), (5.1 + c2 / 2.0, 30.2), (7.7, 52.3), (2.2, 40.0)])
    both = (cubic[0][:2] + [W.QUAD, W.CUBIC, W.LINE], cubic[1] + [(31.2 + c2 / 3.0, 70.0), (33.0, 81.0),
                                                                (33.0 + k / 2, 90.0), (20.0, 95.0), (14.0, 99.0), (1.0, 3.0)])
    _check(gpu_ctx, [cubic, quad, both, quad])


@pytest.mark.parametrize("n", [1, 63, 64, 65, 300, 1000])
def test_paths_of_few_commands(gpu_ctx, n):
    rng = np.random.default_rng(n)
    paths = []
    for _ in range(n):
        v = [[], [W.MOVE], [W.MOVE, W.LINE], [W.MOVE, W.LINE, W.QUAD], [W.LINE, W.LINE]][int(rng.integers(0, 5))]
        paths.append((v, rng.random((int(W.VERB_POINTS[np.array(v, int)].sum()), 2)) * 40.0))
    paths.append(([W.MOVE] + [W.LINE] * n + [W.CLOSE], rng.random((n + 1, 2)) * 90.0))
    _check(gpu_ctx, paths)
