"""The one-wave adjoint over its chunks of 16 and 32 tiles: lines that lie in one
chunk, that cross all of them (a box's sides, closing lines) and that end on a
chunk's last row, tile counts around a chunk and up to the 256 of a path; each
gradient element against the f64 oracle: its adjoint, or, where a vertex lies
exactly on a pixel corner and the oracle's adjoint takes a side of the tie that is
not its forward's, the forward's one-sided difference quotients (a transform's
elements, which many such vertices share: the sums over the points' gradients)."""
import numpy as np
import pytest

import oracle_ref as O
from ochre_amd import workloads as W
from test_gpu_adjoint import oracle_target, perturbed

pytestmark = pytest.mark.gpu


def _path(w, h, lines, seed):
    """A box of nearly the whole area and one contour of short steps through it."""
    rng = np.random.default_rng(seed)
    box = np.array([[1.3, 1.6], [w - 1.4, 2.1], [w - 1.2, h - 1.7], [1.4, h - 1.2]])
    p = np.cumsum(rng.uniform(-6.0, 6.0, (lines + 1, 2)), axis=0)
    p = np.abs((p + 0.5 * np.array([w, h])) % (2.0 * np.array([w, h])) - np.array([w, h])) * 0.94 + 0.5
    p[::7] = np.floor(p[::7] / 8.0) * 8.0  # ends on tile corners: ties of the walk
    return ([W.MOVE] + [W.LINE] * 3 + [W.CLOSE] + [W.MOVE] + [W.LINE] * lines + [W.CLOSE],
            np.concatenate([box, p]).astype(np.float32))


@pytest.mark.parametrize("w,h,lines", [
    (30.0, 30.0, 20), (38.0, 30.0, 60), (62.0, 30.0, 63), (62.0, 38.0, 64),  # 16, 20, 32 and 40 tiles' area
    (62.0, 62.0, 150), (118.0, 118.0, 400),                                  # 64 and 225
    (230.0, 14.0, 130), (14.0, 230.0, 130),                                  # chunks within a row, many rows in a chunk
])
def test_adjoint_over_chunks(gpu_ctx, w, h, lines):
    paths = [_path(w, h, lines, int(10 * w + h) + k) for k in range(3)]
    b = W.from_paths(paths, np.array([[1, 0, 0, 1, 3.7, 5.2], [1, 0, 0, 1, 40.0, -8.0], [0.8, 0.1, -0.2, 1, 9.5, 77.25]],
                                     np.float32))
    tgt, targets = oracle_target(gpu_ctx, perturbed(b, 0.5, 11))
    import torch
    from ochre_amd.device import coverage_adjoint, upload
    loss, dp, dx = (x.cpu().numpy() for x in coverage_adjoint(gpu_ctx, upload(b), tgt))
    torch.cuda.synchronize()
    for i in range(b.n_paths):
        v, p, wt, xf = b.path(i)
        xf = xf.astype(np.float64)
        x0 = np.concatenate([p.astype(np.float64).reshape(-1), xf])
        f = lambda x: O.path_loss64(v, x[:-6].reshape(-1, 2), wt, x[-6:], targets[i])[1]  # noqa: E731
        st, L, gp, gx, _ = O.path_loss64(v, p.astype(np.float64), wt, xf, targets[i], grad=True)
        assert st == 0 and abs(loss[i] - L) <= 1e-3 * max(L, 1.0)
        ref = np.concatenate([gp.reshape(-1), gx])
        got = np.concatenate([dp[b.point_off[i]:b.point_off[i + 1]].reshape(-1), dx[i]])
        tol = 1e-3 * np.maximum(np.abs(ref), 1.0)
        M = xf[:4].reshape(2, 2)
        g = got[:-6].reshape(-1, 2).astype(np.float64) @ np.linalg.inv(M)  # dL/d(world point)
        sums = np.concatenate([(g.T @ p.astype(np.float64)).reshape(-1), g.sum(0)])
        for k in np.nonzero(np.abs(got - ref) > tol)[0]:
            if k >= p.size:
                t = 1e-3 * max(abs(sums[k - p.size]), 1.0)
                assert abs(got[k] - sums[k - p.size]) <= t, (i, k, got[k], ref[k], sums)
                continue
            e = np.zeros_like(x0)
            e[k] = h = 1e-4 / float(xf[0])
            q = sorted([(f(x0 + e) - f(x0)) / h, (f(x0) - f(x0 - e)) / h])
            assert q[0] - tol[k] <= got[k] <= q[1] + tol[k], (i, k, got[k], ref[k], q)
