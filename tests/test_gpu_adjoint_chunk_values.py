"""The one-wave adjoint over its chunks of 16 and 32 tiles, on outlines off
every kink of the loss (no vertex on a tie of the walk): each gradient element
within 1e-3 of the f64 oracle's adjoint, and of nothing else."""
import numpy as np
import pytest

import oracle_ref as O
from ochre_amd import workloads as W
from test_gpu_adjoint import oracle_target, perturbed

pytestmark = pytest.mark.gpu

# area, lines, and three outlines' seeds: the f64 forward's difference quotients of both
# sides agree there for every element, also where a vertex moves by 2e-4 px
CASES = [
    (30.0, 30.0, 20, (1, 1, 1)), (38.0, 30.0, 30, (1, 1, 1)), (62.0, 30.0, 30, (1, 1, 1)),  # 11 to 29 tiles
    (62.0, 38.0, 40, (1, 1, 1)), (62.0, 62.0, 40, (1, 1, 1)),                               # 29 to 48
    (118.0, 118.0, 60, (1, 1, 1)), (180.0, 180.0, 12, (1, 1, 1)),                           # 104 to 168
    (230.0, 14.0, 60, (2, 2, 1)), (14.0, 230.0, 60, (1, 1, 2)),  # chunks within a row, many rows in a chunk
]

TRANSFORMS = np.array([[1, 0, 0, 1, 3.7, 5.2], [1, 0, 0, 1, 40.31, -8.13], [0.8, 0.1, -0.2, 1, 9.5, 77.25]], np.float32)


def outline(w, h, lines, seed):
    p = np.random.default_rng(1000 * seed + lines).uniform(0.03, 0.97, (lines + 1, 2)) * [w, h]
    return [W.MOVE] + [W.LINE] * lines + [W.CLOSE], p.astype(np.float32)


@pytest.mark.parametrize("w,h,lines,seeds", CASES)
def test_adjoint_over_chunks_against_the_oracle(gpu_ctx, w, h, lines, seeds):
    import torch
    from ochre_amd.device import coverage_adjoint, upload
    b = W.from_paths([outline(w, h, lines, k) for k in seeds], TRANSFORMS)
    tgt, targets = oracle_target(gpu_ctx, perturbed(b, 0.5, 11))
    loss, dp, dx = (x.cpu().numpy() for x in coverage_adjoint(gpu_ctx, upload(b), tgt))
    torch.cuda.synchronize()
    for i in range(b.n_paths):
        v, p, wt, xf = b.path(i)
        st, L, gp, gx, _ = O.path_loss64(v, p.astype(np.float64), wt, xf.astype(np.float64), targets[i], grad=True)
        assert st == 0 and abs(loss[i] - L) <= 1e-3 * max(L, 1.0)
        ref = np.concatenate([gp.reshape(-1), gx])
        got = np.concatenate([dp[b.point_off[i]:b.point_off[i + 1]].reshape(-1), dx[i]])
        off = np.abs(got - ref) - 1e-3 * np.maximum(np.abs(ref), 1.0)
        assert off.max() <= 0.0, (i, int(off.argmax()), got[off.argmax()], ref[off.argmax()])
