"""The stage timers' proportions against the kernels' own times, on models of their
own (timing every kernel by itself changes how steps are launched).  Receivers are
a kernel of their own; the tile erosion's time goes to GenerateOrder, Uplift and
Erosion, GenerateOrder also gets a part of the accumulation's.  A sample of steps
stands for the others: tolerance 4 points of the whole, of which the events
around the sampled kernels take up to 2 at the smaller sizes (some 3 us of 150)."""
import subprocess

import numpy as np
import pytest

import fastscape_amd as fa
from conftest import cone_terrain
from test_gpu_parity import CLI, note

pytestmark = pytest.mark.gpu

STAGES = fa.TIMER_NAMES[1:7]


def kernel_shares(m, steps):
    """Shares of the receivers and of the erosion kernels in `steps` steps."""
    m.set_kernel_timing(True)
    before = {k: v[0] for k, v in m.kernel_stats().items()}
    m.step(steps)
    ms = {k: v[0] - before[k] for k, v in m.kernel_stats().items()}
    total = sum(ms.values())
    return ms["k_receivers"] / total, ms["k_tile_erode"] / total


def stage_shares(t):
    total = sum(t[k] for k in STAGES)
    return {k.split(": ")[1]: t[k] / total for k in STAGES}


def check(stages, receivers, erode):
    assert abs(stages["DetermineReceivers"] - receivers) <= 0.04, (stages, receivers)
    order_on = stages["GenerateOrder"] + stages["Uplift"] + stages["Erosion"]
    assert order_on >= erode - 0.04, (stages, erode)
    assert stages["DetermineDonors"] + stages["FlowAcc"] <= 1 - receivers - erode + 0.04


@pytest.mark.parametrize("side", [2048, 4096])
def test_tile_steps(side):
    note("timers %d^2" % side)
    with fa.FastScape(side, side, fa.preset(fa.PRESET_BENCHMARK)) as m:
        m.step(6)
        receivers, erode = kernel_shares(m, 30)
    with fa.FastScape(side, side, fa.preset(fa.PRESET_BENCHMARK)) as m:
        m.step(6)
        m.reset_timers()
        m.step(60)
        check(stage_shares(m.timers()), receivers, erode)


def test_sampled_step_too_deep_for_the_first_halo():
    """25 levels: the first step, sampled, does not erode with the 16-cell halo and
    is taken with the 32-cell one."""
    W, H = 2000, 1600
    note("timers, 25 levels from the first step")
    h = cone_terrain(W, H, 48, 0)
    with fa.FastScape(W, H, fa.preset(fa.PRESET_BENCHMARK), h=h) as m:
        receivers, erode = kernel_shares(m, 1)
    with fa.FastScape(W, H, fa.preset(fa.PRESET_BENCHMARK), h=h) as m:
        m.step(1)
        assert m.tile_stats()["halo32"] == 1
        check(stage_shares(m.timers()), receivers, erode)


def test_every_call_is_accounted_for():
    """Calls of one step, the timers read and reset behind each: every call's stages
    share its time, whichever step was the sample."""
    note("timers of single steps")
    with fa.FastScape(1500, 1100, fa.preset(fa.PRESET_BENCHMARK)) as m:
        m.step(1)
        for i in range(40):
            before = m.timers()
            m.step(1)
            t = m.timers()
            part = np.array([t[k] - before[k] for k in STAGES], float)
            assert part.sum() >= 20, (i, part)      # three kernels of 10 us and more
            assert (part[[0, 1, 2, 3, 5]] > 0).all(), (i, part)
            assert part.sum() <= t["Overall"] - before["Overall"], (i, part)


def test_graph_steps_behind_a_tile_attempt():
    """49 levels: the first step's receivers come from the tile attempts, the later
    ones' are the tile-graph steps' own."""
    W, H, steps = 2000, 1600, 40
    note("timers, 49 levels from the first step")
    h = cone_terrain(W, H, 96, 0)
    with fa.FastScape(W, H, fa.preset(fa.PRESET_BENCHMARK), h=h) as m:
        receivers, _ = kernel_shares(m, steps)
    with fa.FastScape(W, H, fa.preset(fa.PRESET_BENCHMARK), h=h) as m:
        m.step(steps)
        assert m.graph_stats()["steps"] == steps
        share = stage_shares(m.timers())["DetermineReceivers"]
        note("receivers %.4f of the stages, %.4f of the kernels" % (share, receivers))
        assert 0.8 * receivers <= share <= 1.25 * receivers


@pytest.mark.parametrize("path", [fa.PATH_AUTO, fa.PATH_TILE_GRAPH])
def test_depression_filling_is_no_stage(path):
    """Filling takes some ten times as long as a step here; the stages are the
    steps' kernels, the gaps between them and no more."""
    note("timers with depression filling, path %d" % path)
    out = []
    for timing in (True, False):
        with fa.FastScape(700, 501, fa.preset(fa.PRESET_REFERENCE)) as m:
            m.set_path(path)
            m.set_depression_fill(True)
            m.set_kernel_timing(timing)
            m.step(8)
            t = m.timers()
            out.append((sum(v[0] for v in m.kernel_stats().values()) * 1e3,
                        sum(t[k] for k in STAGES), t["Overall"] - t["Step1: Initialize"]))
    kernels, stages, overall = out[0][0], out[1][1], out[1][2]
    note("kernels %.0f us, stages %.0f, overall %.0f" % (kernels, stages, overall))
    assert 0.5 * kernels <= stages <= 2 * kernels


@pytest.mark.parametrize("side,steps", [(101, 60), (1001, 60)])
def test_first_step_of_a_process(tmp_path, side, steps):
    """Loading the kernels takes some 30 ms of a process's first step; that step does
    not stand for the others, whose accumulation and erosion take 20 us or more."""
    note("timers of a process of its own, %d^2" % side)
    r = subprocess.run([CLI, "--preset=benchmark", str(side), str(steps), str(tmp_path / "o.dem"),
                        "1"], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    t = dict(line[2:].split("=")[:2] for line in r.stdout.splitlines() if line.startswith("t "))
    us = {k.strip().split(": ")[-1]: int(v.split()[0]) for k, v in t.items()}
    note("%s" % us)
    assert us["DetermineDonors"] + us["FlowAcc"] + us["GenerateOrder"] + us["Uplift"] + \
        us["Erosion"] >= 10 * steps
    assert us["Uplift"] > 0
