"""A batch of tile steps ends behind a step whose solve fails, wherever in the batch
that is: one cell in a ring at 0 that rises by 1 a step from below, has no receiver
until it is above 0, and then a solve that does not converge."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_parity import note

pytestmark = pytest.mark.gpu

# Newton's iterates of x + keq * x * x = 1.5 end in a cycle
KEQ = float.fromhex("0x1.1fded21c82cafp+3")


@pytest.mark.parametrize("at", [1, 2, 3, 4, 5, 7, 12])
def test_failed_solve_at_a_later_step(at):
    note("solve fails at step %d" % at)
    p = fa.preset(fa.PRESET_REFERENCE, keq=KEQ, dt=1.0, dx=1.0, cell_area=1.0, ueq=1.0,
                  tol=1e-300)
    h = np.zeros((5, 5))
    h[2, 2] = 1.5 - at      # at the step `at`: 0.5, uplifted to 1.5
    ends = []
    for calls in ((40,), (1,) * 40):
        with fa.FastScape(5, 5, p, h=h.ravel()) as m:
            with pytest.raises(fa.FastScapeError) as e:
                for n in calls:
                    m.step(n)
            assert m.path_stats() == {"tile": at, "levels": 0, "graph": 0}
            ends.append((e.value.status, m.getH()))
            assert 0 < ends[-1][1][2, 2] < 1.5
    assert ends[0][0] == ends[1][0]
    np.testing.assert_array_equal(ends[0][1], ends[1][1])
