"""What the batched call hands to the plain pipeline: everything with the dense
kernels off, in bounded passes (a batch over one pass's lines, a single path over
its entries among small ones), equal to the plain call; and with them on the paths
over the largest instance, few or many."""
import numpy as np
import pytest

from ochre_amd import workloads as W
from ochre_amd.device import run_to_host

pytestmark = pytest.mark.gpu


def _glyphs(n):
    return W.glyph_run(n, seed=77)


def _blob_among_glyphs():
    return W.concat([W.glyph_run(150, seed=78), W.star_blobs(n=1, seed=79, nmin=1e5, nmax=1e5, rmin=1950.0, rmax=2000.0),
                     W.glyph_run(149, seed=80)])


@pytest.mark.parametrize("make", [lambda: _glyphs(1), lambda: _glyphs(3), lambda: _glyphs(22000), _blob_among_glyphs],
                         ids=["one", "three", "two passes", "one path over a pass"])
def test_dense_off_equals_plain(gpu_ctx, make):
    b = make()
    cap = b.n_paths * 64 + 400000
    want = run_to_host(gpu_ctx, b, "plain", cap, cap)
    got = run_to_host(gpu_ctx, b, "batched", cap, cap)
    for k, (w, g) in enumerate(zip(want, got)):
        assert np.array_equal(w, g), k


@pytest.mark.parametrize("n_large", [1, 7, 600])
def test_dense_hands_on_large_paths(gpu_ctx, n_large):
    """Paths of about 20 x 20 tiles (over 256 of them) among glyphs: sets exact, alpha within 1 LSB."""
    b = W.concat([W.glyph_run(n_large, seed=81, smin=150.0, smax=170.0), W.glyph_run(40, seed=82)])
    cap = b.n_paths * 500
    want = run_to_host(gpu_ctx, b, "plain", cap, cap)
    got = run_to_host(gpu_ctx, b, "dense", cap, cap)
    for k in (0, 2, 3, 4, 5):
        assert np.array_equal(want[k], got[k]), k
    d = np.abs(want[1].astype(np.int16) - got[1].astype(np.int16))
    assert int(d.max()) <= 1 and float((d != 0).mean()) < 1e-3


@pytest.mark.parametrize("n_first,n_rest,spread", [(2046, 0, 60.0), (2047, 1, 60.0), (3000, 500, 60.0), (2100, 40, 600.0),
                                                   (3000, 3000, 160.0)])
def test_dense_paths_of_many_points(gpu_ctx, n_first, n_rest, spread):
    """Paths over the point count that is tested early: those that fit an instance, and those that
    only their last points put over it."""
    import oracle_ref
    from parity import compare
    rng = np.random.default_rng(n_first + n_rest)
    p = np.concatenate([rng.random((n_first, 2)) * 40.0, rng.random((n_rest, 2)) * spread]).astype(np.float32)
    verbs = [W.MOVE] + [W.LINE] * (len(p) - 1) + [W.CLOSE]
    b = W.concat([W.from_paths([(verbs, p)], np.array([1, 0, 0, 1, 3.25, 7.5], np.float32)), W.glyph_run(5, seed=83)])
    stats = compare(oracle_ref.run_batch(b), run_to_host(gpu_ctx, b, "dense", 20000, 20000), max_lsb=1)
    assert stats["bit_exact_fraction"] >= 0.98  # sums of thousands of increments in arrival order


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257])
def test_dense_few_paths(gpu_ctx, n):
    """Path counts around one per compute unit: sets exact, alpha within 1 LSB of the oracle's."""
    import oracle_ref
    from parity import compare
    b = W.glyph_run(n, seed=90 + n, smin=12.0, smax=110.0)
    stats = compare(oracle_ref.run_batch(b), run_to_host(gpu_ctx, b, "dense", n * 300 + 100, n * 300 + 100), max_lsb=1)
    assert stats["bit_exact_fraction"] >= 0.999
