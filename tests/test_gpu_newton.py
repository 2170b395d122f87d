"""The short form of the Newton solve (a quotient from a refined reciprocal, no
test between iterations) against the oracle's loop, bit for bit, inside its
range and beyond both ends of it: tiny and huge elevations, no uplift, factors
from negligible to far above one, elevations that are no numbers.  On the
halo tiles, the tile graph and the level path."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_parity import note

pytestmark = pytest.mark.gpu

W, H = 97, 70
PATHS = (fa.PATH_AUTO, fa.PATH_TILE_GRAPH, fa.PATH_LEVELS)


def field(scale, seed):
    rng = np.random.default_rng(seed)
    h = rng.random((H, W)) * scale
    h[:2] = h[-2:] = 0
    h[:, :2] = h[:, -2:] = 0
    return np.ascontiguousarray(h).ravel()


def check(oracle, h, which, **kw):
    op = oracle.preset(which, **kw)
    try:
        want = oracle.step(h, W, H, op, oracle.POW_EXACT)["h"]
    except RuntimeError:       # a solve did not converge
        want = None
    for path in PATHS:
        with fa.FastScape(W, H, fa.preset(which, **kw), h=h) as m:
            m.set_path(path)
            if want is None:
                with pytest.raises(fa.FastScapeError):
                    m.step(1)
                continue
            m.step(1)
            np.testing.assert_array_equal(m.getH().ravel(), want, err_msg="path %d" % path)


@pytest.mark.parametrize("scale", [0.0, 1e-310, 1e-200, 2.0 ** -291, 2.0 ** -288, 1e-30, 1.0, 1e6,
                                   2.0 ** 21, 1e30, 2.0 ** 201, 1e200])
def test_linear_solves(oracle, scale):
    note("n = 1, elevations up to %g" % scale)
    for keq in (0.0, 1e-30, 1e-5, 1.0, 1e25, 1e60):
        check(oracle, field(scale, 1), 1, keq=keq)
        check(oracle, field(scale, 2), 1, keq=keq, ueq=0.0, tol=1e-3)
    check(oracle, field(scale, 3), 1, tol=max(scale * 1e-9, 1e-320), ueq=0.0)


@pytest.mark.parametrize("scale", [0.0, 1e-310, 1e-200, 1e-30, 1e-3, 1.0, 1e3, 2.0 ** 20, 2.0 ** 21,
                                   1e9])
def test_square_solves(oracle, scale):
    note("n = 2, elevations up to %g" % scale)
    for keq in (0.0, 1e-30, 2e-6, 1e-3, 1e-1, 10.0):
        check(oracle, field(scale, 4), 0, keq=keq)
        check(oracle, field(scale, 5), 0, keq=keq, ueq=0.0)


def test_values_that_are_no_numbers(oracle):
    note("NaN and infinities")
    for which in (0, 1):
        h = field(1.0, 6)
        h[[500, 1500, 3000]] = np.nan
        h[[700, 2300]] = np.inf
        h[[900, 4100]] = -np.inf
        check(oracle, h, which)
