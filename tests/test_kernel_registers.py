"""The hierarchical fastconv kernels of 8192 points run two workgroups a CU: at
most 128 vector registers and half the LDS each, in interleaved and in split
storage."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "openvsip_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_two_workgroups_a_cu(tmp_path):
    run = subprocess.run([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                          "-packed-fp32-ops", "-ffp-contract=fast", "-w", "--cuda-device-only",
                          "-Rpass-analysis=kernel-resource-usage", "-c", os.path.join(CSRC, "ovx_hier.hip"), "-o",
                          str(tmp_path / "hier.o")], check=True, capture_output=True, text=True)
    used = {}
    for part in run.stderr.split("Function Name: ")[1:]:
        used[part.split()[0]] = (int(re.search(r"\bVGPRs: (\d+)", part).group(1)),
                                 int(re.search(r"LDS Size \[bytes/block\]: (\d+)", part).group(1)))
    kernels = [v for k, v in used.items() if "k_hier_fastconvILi8192E" in k]
    assert len(kernels) == 2
    for registers, lds in kernels:
        assert registers <= 128 and lds <= 80 * 1024
