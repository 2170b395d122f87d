"""An ensemble's schedule lays its work out: sixteen tiles per erosion workgroup are
solved one after another, so 256 tiles, one to a CU, take several times as long
that way.  The search times such differences and keeps the better schedule."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_ensemble import bench, make, note

pytestmark = pytest.mark.gpu

SPECS = [(1024, 1024, bench(), 1)]


def step_ms(ens, sched, steps=40):
    ens.set_schedule(fa.schedule(**sched))
    ens.run(4)
    n0, ms0 = ens.stats()
    ens.run(steps - 1)
    n, ms = ens.stats()
    return (ms - ms0) / (n - n0)


def test_tiles_per_claim_has_an_effect():
    note("tiles per erosion workgroup")
    with make(SPECS) as ens:
        one = step_ms(ens, dict(tiles_per_claim=1))
        sixteen = step_ms(ens, dict(tiles_per_claim=16))
        note("%.1f us a step with one tile, %.1f with sixteen" % (1e3 * one, 1e3 * sixteen))
        assert sixteen >= 2 * one


def test_search_leaves_a_bad_schedule():
    note("search from sixteen tiles per workgroup")
    with make(SPECS) as ens:
        ens.run(4)
        ens.set_schedule(fa.schedule(tiles_per_claim=16))
        ens.autotune(8)
        ens.run(79)
        log = ens.tune_log()
        note("%s" % log)
        assert ens.get_schedule().as_dict()["tiles_per_claim"] < 16


def test_slow_first_steps_pick_no_schedule():
    """A run's first steps are its slowest (code and memory are touched for the first
    time, drainage is new); two tiles a workgroup take half as long again as one."""
    note("search from a fresh start")
    specs = [(160, 160, bench(keq=1e-5 * (1 + i % 7)), i) for i in range(28)]   # 252 tiles
    for _ in range(5):
        with make(specs) as ens:
            ens.autotune(1)
            ens.run(19)
            note("%s" % ens.tune_log())
            assert ens.get_schedule().as_dict()["tiles_per_claim"] == 1


# the last workgroup's share: whole, one item, all but one, and more than there are
@pytest.mark.parametrize("per", [2, 3, 5, 16])
@pytest.mark.parametrize("specs", [
    [(64, 64, bench(), 0)], [(129, 65, bench(), 1), (64, 64, bench(), 2)],
    [(200, 150, bench(), 3), (70, 70, fa.preset(fa.PRESET_REFERENCE), 4), (320, 64, bench(), 5)],
    [(130, 70, fa.preset(fa.PRESET_REFERENCE), 0)]])
def test_shares_of_workgroups(specs, per):
    note("%d realizations, %d tiles a workgroup" % (len(specs), per))
    with make(specs) as base, make(specs) as other:
        other.set_schedule(fa.schedule(recv_rows=min(256, 64 * per), tiles_per_claim=per))
        base.run(20)
        other.run(20)
        for r in range(len(specs)):
            np.testing.assert_array_equal(other.getH(r), base.getH(r), err_msg="r%d" % r)
            np.testing.assert_array_equal(other.accum(r), base.accum(r), err_msg="r%d" % r)
