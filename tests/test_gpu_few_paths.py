"""Batches of at most one path per compute unit, which the 16-wave dense instance
takes alone: what it must not hand on."""
import numpy as np
import pytest

import oracle_ref
from ochre_amd import workloads as W
from parity import compare

pytestmark = pytest.mark.gpu


def _scribble(n, reach, seed):
    """n cubics within `reach` px."""
    rng = np.random.default_rng(seed)
    p = rng.uniform(0.0, reach, (3 * n + 1, 2))
    return [W.MOVE] + [W.CUBIC] * n + [W.CLOSE], p.astype(np.float32)


def _handed_on(ctx, b, mode="dense"):
    """The output, and how many passes the plain pipeline made for handed-on paths."""
    from ochre_amd.device import run_to_host
    ctx.set_timing(True)
    try:
        got = run_to_host(ctx, b, mode, 8192, 8192)
        return got, ctx.timing("pass.lines")[1]
    finally:
        ctx.set_timing(False)


@pytest.mark.parametrize("n,reach", [(1000, 40.0), (900, 100.0), (2100, 40.0)])
def test_paths_of_many_curves_stay_in_the_dense_kernel(gpu_ctx, n, reach):
    """More lines than 256 commands of a path may have, spread over more commands than that."""
    b = W.from_paths([_scribble(n, reach, n + int(reach))], np.array([1, 0, 0, 1, 11.3, 6.7], np.float32))
    lines = oracle_ref.run_batch(b).stats["lines"]
    assert 8192 < lines < 8192 * n / 256, lines
    got, passes = _handed_on(gpu_ctx, b)
    assert passes == 0
    stats = compare(oracle_ref.run_batch(b), got, max_lsb=1)
    assert stats["bit_exact_fraction"] >= 0.98  # sums of thousands of increments in arrival order
