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
