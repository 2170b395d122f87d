"""The halo cells that drain into a tile: none, a few, as many as a wave's share
of the list holds and far more (valleys whose whole flanks drain into one
tile), on both halo sizes, at grid edges and on ragged tiles.  The same bits as
the level path, which has no tiles."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_parity import note

pytestmark = pytest.mark.gpu


def valleys(W, H, period, at, axis, skew, tilt):
    """Straight flanks down to valley lines `period` apart; with skew the
    flanks run diagonally.  The valleys' floors are outlets all along, or with
    tilt rivers to the grid's edge (too long for the halo)."""
    y, x = np.mgrid[0:H, 0:W].astype(np.float64)
    u, v = (x, y) if axis == 0 else (y, x)
    if skew:
        u = u + v
    d = np.abs((u - at + period / 2) % period - period / 2)
    h = 1.0 + d + tilt * v
    h[:2] = h[-2:] = 0
    h[:, :2] = h[:, -2:] = 0
    return np.ascontiguousarray(h).ravel()


@pytest.mark.parametrize("tilt", [0.0, 1e-7])
@pytest.mark.parametrize("axis,skew", [(0, False), (1, False), (0, True)])
@pytest.mark.parametrize("period", [4, 12, 27, 50])
@pytest.mark.parametrize("W,H", [(160, 140), (129, 133), (70, 200)])
def test_inflow_from_the_halo(W, H, period, axis, skew, tilt):
    note("valleys %dx%d every %d, axis %d" % (W, H, period, axis))
    for at in (62, 65):   # just inside the first tile, just outside
        h = valleys(W, H, period, at, axis, skew, tilt)
        out = []
        for path in (fa.PATH_AUTO, fa.PATH_LEVELS):
            with fa.FastScape(W, H, fa.preset(fa.PRESET_BENCHMARK), h=h) as m:
                m.set_path(path)
                m.step(2)
                out.append((m.getH(), m.path_stats()))
        np.testing.assert_array_equal(out[0][0], out[1][0])
        # the halo tiles take the step unless a tile's chains need more halo
        # cells than they hold (flanks of 13 cells that drain out of a tile do)
        if axis == 0 and not skew and not tilt and (period <= 12 or (period == 27 and W == 70)):
            assert out[0][1]["tile"] == 2
