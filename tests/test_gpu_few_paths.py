"""Batches of at most one path per compute unit, which the 16-wave dense instance
takes alone: what it must not hand on, and what tuning on such a batch leaves as it
was."""
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


def test_tuning_on_few_paths_leaves_the_shapes(gpu_ctx):
    """The 64-tile and small-grid shapes are not used by such a batch, so timing it must
    not choose them; each configuration reported is one that the call can take."""
    from ochre_amd.device import (Context, DeviceOutput, autotune, dense_params, set_dense_params, set_dense_small,
                                  upload)
    ctx = Context(0)
    try:
        set_dense_params(ctx, True, 3, 2)
        set_dense_small(ctx, 6)
        was = dense_params(ctx)
        b = W.glyph_run(61, seed=3)
        _, results = autotune(ctx, upload(b), DeviceOutput(b.n_paths, 8192, 8192), reps=1)
        assert dense_params(ctx) == was
        shapes = [tuple(v for k, v in sorted(r.items()) if k.startswith("dense")) for r in results]
        assert len(set(shapes)) == len(shapes) == 1
    finally:
        ctx.close()


def test_tuning_key_tells_the_two_routes_apart(gpu_ctx, tmp_path):
    """As many paths as compute units and a few more lie in one power of two; only the
    second batch uses the tuned shapes."""
    import torch
    from ochre_amd.device import (Context, DeviceOutput, autotune_cached, dense_params, set_dense_large, set_dense_params,
                                  set_dense_small, upload)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    if (cus + 1).bit_length() != cus.bit_length():
        pytest.skip("one more path is another power of two")
    path = str(tmp_path / "tune.txt")
    ctx = Context(0)
    try:
        for n in (cus, cus + 1):
            # the same path n times: mean commands and points alike
            one = W.glyph_run(1, seed=41)
            b = one.subset([0] * n)
            assert autotune_cached(ctx, upload(b), DeviceOutput(n, 128 * n, 128 * n), reps=1, cache_path=path), n
        tuned = dense_params(ctx)
        assert len(open(path).read().splitlines()) == 2
        # found again: the first one leaves what the context has, the second sets the shapes
        set_dense_large(ctx, True)  # (tuning the second may have chosen otherwise)
        set_dense_params(ctx, True, 3, 2)
        set_dense_small(ctx, 6)
        mine = dense_params(ctx)
        for n in (cus, cus + 1):
            b = one.subset([0] * n)
            assert not autotune_cached(ctx, upload(b), DeviceOutput(n, 128 * n, 128 * n), reps=1, cache_path=path), n
            if n == cus:
                assert dense_params(ctx) == mine
        assert dense_params(ctx) == tuned
    finally:
        ctx.close()


def test_tuning_on_few_paths_without_the_large_instance(gpu_ctx):
    """Then such a batch does use the shapes, and they are timed as for any other."""
    from ochre_amd.device import Context, DeviceOutput, autotune, dense_params, set_dense_large, upload
    ctx = Context(0)
    try:
        set_dense_large(ctx, False)
        b = W.glyph_run(61, seed=3)
        best, results = autotune(ctx, upload(b), DeviceOutput(b.n_paths, 8192, 8192), reps=1)
        assert len(results) == 10 + 4 + 2
        assert all(dense_params(ctx)[k] == best[k] for k in ("dense_groups_per_cu", "dense_waves_per_group"))
    finally:
        ctx.close()
