"""The receivers kernel (64 columns x 6 rows per wave) at the edges of its
blocks, against the oracle's ComputeReceivers: one interior cell, one row or
column group more or less than a wave or workgroup holds, long thin grids, and
terrains with many ties (whole-number elevations), whose receivers need the
divisions.  Receivers are whole numbers: exactly equal."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_parity import gpu_params, note, oracle_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(5, 5), (67, 9), (68, 10), (69, 11), (130, 27), (132, 28),
                                 (133, 29), (1500, 6), (6, 1500)])
def test_receivers_at_block_edges(oracle, W, H):
    note("receivers %dx%d" % (W, H))
    rng = np.random.default_rng(W * H)
    for preset in (0, 1):
        op = oracle_params(oracle, preset)
        for ties in (False, True):
            h = rng.random(W * H) if not ties else rng.integers(0, 4, W * H).astype(float)
            with fa.FastScape(W, H, gpu_params(preset), h=h) as m:
                m.step(1)
                np.testing.assert_array_equal(m.receivers(), oracle.receivers(h, W, H, op))
