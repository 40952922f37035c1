"""The batched call's captured graph: captured where a call repeats the arguments of
the one before, replayed while they stay, captured again after they change; every
call checked against the oracle, with eager work and a synchronisation between, and
the replays counted."""
import numpy as np
import pytest

import oracle_ref
from ochre_amd import workloads as W
from parity import compare

pytestmark = pytest.mark.gpu

SHAPES = [(4, 4, 0, 1), (2, 2, 0, 0), (4, 4, 8, 1), (2, 8, 0, 1), (1, 4, 4, 0)]  # groups, waves, small, large


def _large(seed):
    return W.glyph_run(2, seed=seed, smin=150.0, smax=170.0)  # over every dense instance


@pytest.mark.parametrize("groups,waves,small,large", SHAPES)
@pytest.mark.parametrize("n", [40, 700])
def test_replays_give_the_oracles_result(gpu_ctx, n, groups, waves, small, large):
    import torch
    from ochre_amd.device import (Context, DeviceOutput, rasterize_batched, set_dense_large, set_dense_params,
                                  set_dense_small, upload)
    ctx = Context(0)
    try:
        set_dense_params(ctx, True, groups, waves)
        set_dense_small(ctx, small)
        set_dense_large(ctx, bool(large))
        calls = []
        for seed in (9, 10):
            b = W.concat([W.glyph_run(n=n, seed=seed), W.random_paths(30, seed), _large(seed)])
            ref = oracle_ref.run_batch(b)
            calls.append((ref, upload(b), DeviceOutput(b.n_paths, ref.n_tiles + 16, ref.n_spans + 16)))

        def call(k):
            ref, db, out = calls[k]
            for t in (out.tile_xy, out.tile_alpha, out.span_xy, out.span_w, out.path_tile_count, out.path_span_count):
                t.zero_()
            rasterize_batched(ctx, db, out)
            torch.cuda.synchronize()
            st = compare(ref, out.to_host(), max_lsb=1)
            assert st["bit_exact_fraction"] >= 0.999
            _ = (torch.rand(1000, device="cuda") * 2.0).sum().item()

        def replays(order):
            ctx.set_timing(True)
            for k in order:
                call(k)
            return ctx.timing("batched_graph")[1]

        assert replays([0]) == 0  # new arguments: the launches themselves
        assert replays([0, 0, 0]) == 3  # captured, then replayed
        assert replays([1, 0]) == 1  # others, then the captured ones again
        assert replays([1, 1, 1]) == 2  # captured anew
        assert replays([0, 1]) == 1
        assert replays([0, 0]) == 1
    finally:
        ctx.close()
