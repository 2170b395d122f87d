"""Grids of at least four tiles per CU, whose accumulation runs on 512 threads a
tile: rows of every alignment with dwords cut at the last column, natural drainage
and valleys whose flanks overflow a wave's share of the inflow list (33 ring cells
with five halo cells behind each of them; the share holds 128).  The same bits as
the level path."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_inflow import valleys
from test_gpu_parity import note

pytestmark = pytest.mark.gpu


def compare(W, H, h):
    out = []
    for path in (fa.PATH_AUTO, fa.PATH_LEVELS):
        with fa.FastScape(W, H, fa.preset(fa.PRESET_BENCHMARK), h=h) as m:
            m.set_path(path)
            m.step(2)
            out.append((m.getH(), m.accum(), m.path_stats()["tile"]))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
    assert out[0][2] == 2


@pytest.mark.parametrize("W", [2113, 2114, 2115])
def test_natural_drainage(W):
    H = 2050
    note("%dx%d" % (W, H))
    with fa.FastScape(W, H, fa.preset(fa.PRESET_BENCHMARK)) as m:
        m.step(40)
        h = np.ascontiguousarray(m.getH()).ravel()
    compare(W, H, h)


@pytest.mark.parametrize("W,axis", [(2113, 0), (2114, 1), (2115, 0)])
def test_valleys_overflow_the_list(W, axis):
    H = 2050
    note("valleys %dx%d axis %d" % (W, H, axis))
    compare(W, H, valleys(W, H, 12, 65, axis, False, 0.0))
