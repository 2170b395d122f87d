"""Registers of kernels whose residency depends on them.  A 1024-thread workgroup
is four waves a SIMD, so two on a CU need eight waves' registers there: up to 64
vector and 80 scalar ones each (of 800, in blocks of 16, with the 16 of the trap
handler)."""
import os
import re
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "barnes2019-landscape_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


# k_tile_erode<n, timed> with both halos; k_ens_erode<n, many>
@pytest.mark.parametrize("source,kernel,count", [
    ("fastscape_hip.hip", "k_tile_erode", 8), ("fs_ensemble.hip", "k_ens_erode", 4)])
def test_two_erosion_workgroups_per_cu(tmp_path, source, kernel, count):
    r = subprocess.run(
        [HIPCC, "-O3", "-std=c++17", "-ffp-contract=off", "-w", "--offload-arch=gfx950", "-Xclang",
         "-target-feature", "-Xclang", "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"),
         "-I" + CSRC, "--cuda-device-only", "-S", os.path.join(CSRC, source), "-o",
         str(tmp_path / "out.s"), "-Rpass-analysis=kernel-resource-usage"],
        check=True, capture_output=True, text=True)
    used = {}
    for part in r.stderr.split("Function Name: ")[1:]:
        if re.match(r"\S*" + kernel + r"ILi[12]ELb[01]E", part):
            used[part.split()[0]] = tuple(int(re.search(k + r": (\d+)", part).group(1))
                                          for k in (r"\bVGPRs", "TotalSGPRs"))
    assert len(used) == count, used
    assert all(v <= 64 and s <= 80 for v, s in used.values()), used
