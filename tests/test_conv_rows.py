"""Offsets of the small-level convolution into its input rows, on images beyond
the reach of 32-bit offsets (csrc/fs_conv_rows.h, run on the CPU)."""
import os
import subprocess

from conftest import ROOT

CSRC = os.path.join(ROOT, "barnes2019-landscape_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_offsets_equal_those_of_64_bits(tmp_path):
    exe = tmp_path / "rows"
    subprocess.run([HIPCC, "-O1", "-std=c++17", "-I" + CSRC,
                    os.path.join(ROOT, "tests", "native", "conv_rows_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True)
    rows, bad, far = map(int, subprocess.run([str(exe)], check=True, capture_output=True,
                                             text=True).stdout.split())
    assert rows > 20000 and far > 1000 and bad == 0
