"""Where the Newton loop ends: an infinite tolerance lets it take no iteration at
all, the oracle's bits on every path."""
import pytest

from test_gpu_newton import check, field
from test_gpu_parity import note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", [0, 1])
def test_infinite_tolerance(oracle, which):
    note("infinite tolerance, preset %d" % which)
    check(oracle, field(1.0, 7), which, tol=float("inf"))
