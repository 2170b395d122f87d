"""The fill kernel at the edges of its 64 x 64 tiles and 16 x 16 wave patches,
with the paths that cross them: a serpentine channel through every patch, flats
and whole-number ties, negative elevations, signed zeros and an infinite peak.
The oracle's priority-flood gives the same bits."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_fill import note

pytestmark = pytest.mark.gpu


def terrain(kind, W, H):
    rng = np.random.default_rng(W * 1000 + H)
    if kind == "ties":
        h = rng.integers(-2, 3, (H, W)).astype(np.float64)
    elif kind == "negative":
        h = rng.normal(-1.0, 1.0, (H, W))
        h[rng.random((H, W)) < 0.1] = -0.0
        h[H // 2, W // 2] = np.inf
    else:
        # walls every other row with one gap each, alternating sides: the
        # channel's floor is below its outlet
        h = np.full((H, W), 1.0)
        h[::2] = 9.0
        h[2:-2:4, 2] = 1.0
        h[4:-2:4, W - 3] = 1.0
        h[0:2] = h[-2:] = 5.0
    return np.ascontiguousarray(h).ravel()


@pytest.mark.parametrize("kind", ["ties", "negative", "serpentine"])
@pytest.mark.parametrize("W,H", [(5, 6), (17, 19), (64, 66), (65, 63), (129, 80), (66, 200)])
def test_fill_at_tile_and_patch_edges(oracle, W, H, kind):
    note("fill %s %dx%d" % (kind, W, H))
    h = terrain(kind, W, H)
    with fa.FastScape(W, H, fa.preset(fa.PRESET_BENCHMARK), h=h) as m:
        m.fill_depressions()
        np.testing.assert_array_equal(m.getH().ravel(), oracle.fill_depressions(h, W, H))
