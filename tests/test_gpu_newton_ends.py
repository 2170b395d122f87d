"""Where the Newton loop ends: an infinite tolerance lets it take no iteration at
all (the oracle's bits), and a solve that takes its hundredth iteration has
failed, even where that one converges, on every path."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_newton import PATHS, check, field
from test_gpu_parity import note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", [0, 1])
def test_infinite_tolerance(oracle, which):
    note("infinite tolerance, preset %d" % which)
    check(oracle, field(1.0, 7), which, tol=float("inf"))


# one interior cell h0 among cells at hn, fact = keq: the 99th iterate differs
# from the 98th, the 100th from the 99th by nothing
@pytest.mark.parametrize("h0,hn,keq", [
    ("0x1.937eff33d6419p-1", "-0x1.54a31ad1048d2p-1", "0x1.d1e552113bc0ep+0"),
    ("0x1.64a945552e70ep-14", "-0x1.5bc7bb432d1b3p-14", "0x1.7e389882ccd72p+13")])
def test_hundredth_iteration(h0, hn, keq):
    note("100 iterations from " + h0)
    h0, hn, keq = (float.fromhex(v) for v in (h0, hn, keq))
    kw = dict(keq=keq, dt=1.0, dx=1.0, cell_area=1.0, ueq=0.0, tol=1e-300)
    h = np.full((5, 5), hn)
    h[2, 2] = h0
    h = h.ravel()
    for path in PATHS:
        with fa.FastScape(5, 5, fa.preset(0, **kw), h=h) as m:
            m.set_path(path)
            with pytest.raises(fa.FastScapeError):
                m.step(1)
