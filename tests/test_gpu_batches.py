"""Tile steps are launched in batches; a batch ends early where drainage gets
too deep for the halo, or shallow enough for the smaller one.  One call of
many steps gives the bits, the receivers and counts of the last step, and the
path of every step, that as many calls of one step give."""
import numpy as np
import pytest

import fastscape_amd as fa
from conftest import cone_terrain
from test_gpu_parity import gpu_params, note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,preset,steps,kind", [
    (101, 67, 1, 1, "random"), (101, 67, 1, 4, "random"), (130, 70, 1, 77, "random"),
    (300, 260, 0, 40, "random"),        # 16-cell halo, 32-cell halo, tile graph
    (257, 190, 0, 9, "random"),
    (200, 160, 1, 70, "cone"),          # 25 levels deep from the first step
    (640, 400, 1, 420, "random")])      # drainage around 16 levels: both halos in turn
def test_one_call_equals_single_steps(oracle, W, H, preset, steps, kind):
    note("batches %dx%d preset %d, %d steps" % (W, H, preset, steps))
    h0 = oracle.init_terrain(W, H, 0) if kind == "random" else cone_terrain(W, H, 48, 0)
    with fa.FastScape(W, H, gpu_params(preset), h=h0) as a, \
            fa.FastScape(W, H, gpu_params(preset), h=h0) as b:
        a.step(steps)
        for _ in range(steps):
            b.step(1)
        assert a.path_stats() == b.path_stats() and a.tile_stats() == b.tile_stats()
        np.testing.assert_array_equal(a.getH(), b.getH())
        np.testing.assert_array_equal(a.receivers(), b.receivers())
        np.testing.assert_array_equal(a.accum(), b.accum())
        np.testing.assert_array_equal(a.levels(), b.levels())
        t = a.timers()
        assert sum(t[k] for k in fa.TIMER_NAMES[1:7]) <= t["Overall"], t


def test_failed_solve_ends_the_batch():
    """The step whose Newton solve fails is the last one taken."""
    note("failed solve in a batch")
    p = fa.preset(fa.PRESET_REFERENCE, tol=1e-300)
    ends = []
    for calls in ((20,), (1,) * 20):
        with fa.FastScape(64, 64, p, engine_seed=2) as m:
            err = None
            for n in calls:
                try:
                    m.step(n)
                except fa.FastScapeError as e:
                    err = e
                    break
            ends.append((err and err.status, m.path_stats(), m.getH()))
    assert ends[0][0] == ends[1][0]
    if ends[0][0] is not None:
        assert ends[0][1] == ends[1][1]
        np.testing.assert_array_equal(ends[0][2], ends[1][2])
