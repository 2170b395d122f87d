"""The network's host code on the CPU, against a HIP runtime of stand-ins
(native/unet_host_check.cpp)."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "barnes2019-landscape_amd", "csrc")
INCLUDE = os.path.join(ROOT, "include")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    """Runs the program; its output's lines as lists of words."""
    d = tmp_path_factory.mktemp("unet_host")
    host = [HIPCC, "-O1", "-std=c++17", "-fPIC", "-w", "-I" + INCLUDE, "-I" + CSRC, "-x", "hip",
            "--cuda-host-only", "-c"]
    objs = []
    for src in (os.path.join(CSRC, "fs_unet.hip"), os.path.join(CSRC, "fs_host.cpp"),
                os.path.join(ROOT, "tests", "native", "unet_host_check.cpp")):
        objs.append(str(d / (os.path.basename(src) + ".o")))
        subprocess.run(host + [src, "-o", objs[-1]], check=True, capture_output=True)
    # the device code's image stays unresolved: nothing is launched
    subprocess.run(["g++", *objs, "-o", str(d / "check"), "-lpthread",
                    "-Wl,--unresolved-symbols=ignore-all"], check=True, capture_output=True)

    def run(*args):
        r = subprocess.run([str(d / "check"), *map(str, args)], capture_output=True, text=True,
                           timeout=100)
        assert r.returncode == 0, r.stderr
        return [line.split() for line in r.stdout.splitlines()]
    return run


@pytest.mark.parametrize("H,W,max_batch", [
    (352, 352, 32), (448, 480, 16), (256, 352, 32), (352, 480, 64), (32, 32, 256), (256, 256, 32)])
def test_every_batch_has_its_workspace(check, H, W, max_batch):
    """The partial sums of a smaller batch can need more chunks than those of
    the largest."""
    assert check("batches", H, W, max_batch) == [[str(max_batch)]]


def test_a_failed_call_waits_for_its_copies(check):
    """Whichever runtime call of loss_grad fails, no copy to or from the caller's
    arrays is left behind, and the failure is reported."""
    left = check("failures", 64, 64, 4)
    assert left[:-1] == []
    assert int(left[-1][0]) > 60
