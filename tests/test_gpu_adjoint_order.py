"""The adjoint of more paths than it has waves, whose queue runs the longest paths
first: losses and gradients are those of the same paths in smaller calls, bit for
bit (the handed-on path, whose sums are atomic, to 1e-4), with empty paths, a point, a zero transform, a path that is handed on and
lengths from under a pixel to hundreds among them."""
import numpy as np
import pytest

from ochre_amd import workloads as W

pytestmark = pytest.mark.gpu


def _paths(n, seed):
    rng = np.random.default_rng(seed)
    v, xf = [], []
    for i in range(n):
        k = int(rng.integers(3, 9))
        verbs, pts = [W.MOVE] + [W.LINE] * (k - 1) + [W.CLOSE], rng.random((k, 2))
        s = float(2.0 ** rng.uniform(-2.0, 6.5))
        if i % 401 == 7:
            verbs, pts = [], np.zeros((0, 2))
        if i % 401 == 8:
            verbs, pts = [W.MOVE, W.CLOSE], pts[:1]
        if i % 401 == 9:
            s = 0.0
        if i == n // 2:
            s = 600.0  # over a wave's 32 x 32-tile grid
        v.append((verbs, pts.astype(np.float32)))
        xf.append([s, 0, 0, s, rng.uniform(0, 64), rng.uniform(0, 64)])
    return v, np.array(xf, np.float32)


@pytest.mark.parametrize("n", [2048, 2049, 3001])
def test_order_changes_nothing(gpu_ctx, n):
    import torch
    from ochre_amd.device import DeviceOutput, coverage_adjoint, rasterize_plain, upload
    v, xf = _paths(n, n)

    def run(lo, hi):
        b = W.from_paths(v[lo:hi], xf[lo:hi])
        t = W.from_paths(v[lo:hi], xf[lo:hi] * np.float32(1.03))
        out = DeviceOutput(hi - lo, 200000, 100000, coverage=True)
        rasterize_plain(gpu_ctx, upload(t), out)
        r = [x.cpu().numpy() for x in coverage_adjoint(gpu_ctx, upload(b), out)]
        torch.cuda.synchronize()
        return r

    whole, parts = run(0, n), [run(lo, min(n, lo + 1000)) for lo in range(0, n, 1000)]
    m, off = n // 2, np.cumsum([0] + [len(p) for _, p in v])
    for k, big in enumerate([slice(m, m + 1), slice(2 * off[m], 2 * off[m + 1]), slice(6 * m, 6 * m + 6)]):
        got, ref = whole[k].reshape(-1), np.concatenate([p[k].reshape(-1) for p in parts])
        assert np.allclose(got[big], ref[big], rtol=1e-4, atol=1e-4)
        got[big] = ref[big]
        assert np.array_equal(got, ref)
