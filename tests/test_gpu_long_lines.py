"""Lines of 3,000 to 58,000 px through the batched call's unordered tile stage:
near-diagonal ribbons and polygons, whose f32 crossing parameters drift up to many
pixels from the line, so that an increment's area is far over a pixel's.  Sets
exact, alpha within 1 LSB of the oracle's."""
import numpy as np
import pytest

import oracle_ref
from ochre_amd import workloads as W
from parity import compare

pytestmark = pytest.mark.gpu


def _ribbon(length, slope=0.989, width=0.5):
    """A strip `width` px wide along a line of `length` px (longer axis) through the origin."""
    h = 0.5 * length
    return np.array([(-h, -h * slope), (h, h * slope), (h + width, h * slope), (-h + width, -h * slope)], np.float32)


def _polygon(n, reach, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(-reach, reach, (n, 2)).astype(np.float32)


PATHS = {
    # 4 lines of 29,000 px
    "ribbon given": np.array([(-14499.7, -14339.8), (14499.8, 14340.1), (14500.3, 14340.1), (-14499.2, -14339.8)], np.float32),
    "ribbon 3000": _ribbon(3000.3),
    "ribbon 4080": _ribbon(4080.7, 0.9995),
    "ribbon 4096": _ribbon(4096.0, 0.9995),
    "ribbon 4097": _ribbon(4097.0, 0.9995),
    "ribbon 12000": _ribbon(12000.9, 0.998),
    "ribbon 20000": _ribbon(20000.3),
    "ribbon 50000": _ribbon(50000.3, 0.9991),
    "ribbon 50000 wide": _ribbon(50000.3, -0.9991, 3.0),
    # tall and narrow, wide and flat: one side of the grid short
    "tall": np.array([(-1500.2, -29000.4), (1500.9, 29000.3), (1501.6, 29000.3), (-1499.5, -29000.4)], np.float32),
    "flat": np.array([(-29000.4, -1500.2), (29000.3, 1500.9), (29000.3, 1501.6), (-29000.4, -1499.5)], np.float32),
    "polygon 7": _polygon(7, 16000.0, 3),
}


@pytest.mark.parametrize("name", list(PATHS))
def test_long_lines_dense(gpu_ctx, name):
    from ochre_amd.device import run_to_host
    p = PATHS[name]
    b = W.from_paths([([W.MOVE] + [W.LINE] * (len(p) - 1) + [W.CLOSE], p)], W.IDENTITY)
    ref = oracle_ref.run_batch(b)
    print(f"[long lines] {name}: {ref.n_tiles} tiles", flush=True)
    st = compare(ref, run_to_host(gpu_ctx, b, "dense", ref.n_tiles + 64, ref.n_spans + 64), max_lsb=1)
    print(f"[long lines] {name}: {st}", flush=True)
    assert st["bit_exact_fraction"] >= 0.995


def test_long_lines_coverage(gpu_ctx):
    """The f32 coverage of the same stage against the ordered one's: a saturated
    sum is off by up to 0.1, a regrouped one by rounding."""
    import torch
    from ochre_amd.device import DeviceOutput, rasterize_batched, rasterize_plain, upload
    p = PATHS["ribbon given"]
    b = W.from_paths([([W.MOVE] + [W.LINE] * (len(p) - 1) + [W.CLOSE], p)], W.IDENTITY)
    covs = []
    for run in (rasterize_plain, rasterize_batched):
        out = DeviceOutput(1, 20000, 20000, coverage=True)
        run(gpu_ctx, upload(b), out)
        torch.cuda.synchronize()
        covs.append(out.tile_cov[:out.n_tiles].cpu().numpy())
    assert covs[0].shape == covs[1].shape
    # a pixel of 4 lines has at most 8 increments of up to 16, and its carry as many
    # heights as a row of the ribbon: some 40 f32 roundings of values below 16
    assert float(np.abs(covs[0] - covs[1]).max()) <= 40 * 16 * 2.0 ** -24
