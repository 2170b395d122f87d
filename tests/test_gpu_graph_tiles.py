"""The tile graph at tile counts around its 64 groups and work queues: one tile,
one short of a group each, one each, one over, two rounds; after a model of
another size, so that device memory comes back used.  The same bits as the
level path, whose steps share none of the graph's kernels."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_parity import note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", [fa.PRESET_REFERENCE, fa.PRESET_BENCHMARK])
@pytest.mark.parametrize("tx,ty", [(1, 1), (9, 7), (8, 8), (13, 5), (32, 4), (13, 10)])
def test_tile_counts(which, tx, ty):
    W, H = 64 * tx, 64 * ty - 3
    note("%d tiles, preset %d" % (tx * ty, which))
    with fa.FastScape(W, H, fa.preset(which)) as m:
        m.step(30)
        h = np.ascontiguousarray(m.getH()).ravel()
    out = []
    for path in (fa.PATH_TILE_GRAPH, fa.PATH_LEVELS):
        with fa.FastScape(W, H, fa.preset(which), h=h) as m:
            m.set_path(path)
            m.step(3)
            out.append(m.getH())
    np.testing.assert_array_equal(out[0], out[1])
