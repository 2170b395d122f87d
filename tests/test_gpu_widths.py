"""Rows of every alignment: widths over two residues modulo 4 and more, inner
tiles and those at the grid's edges, on both halo sizes.  The same bits as the
level path."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_parity import note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(193, 200), (194, 150), (195, 201), (196, 97), (209, 193),
                                 (65, 70), (63, 66), (67, 5), (5, 67), (257, 255)])
def test_widths(W, H):
    note("%dx%d" % (W, H))
    with fa.FastScape(W, H, fa.preset(fa.PRESET_BENCHMARK)) as m:
        fields = []
        for n in (1, 40, 250):   # fresh, shallow, deep drainage
            m.step(n)
            fields.append(np.ascontiguousarray(m.getH()).ravel())
    for h in fields:
        out = []
        for path in (fa.PATH_AUTO, fa.PATH_LEVELS):
            with fa.FastScape(W, H, fa.preset(fa.PRESET_BENCHMARK), h=h) as m:
                m.set_path(path)
                m.step(2)
                out.append(m.getH())
        np.testing.assert_array_equal(out[0], out[1])
