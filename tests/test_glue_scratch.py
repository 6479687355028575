"""The scratch of a half-row solve's last step (words of more strands than are listed,
oneesan-gpu_amd/csrc/ofp_glue_impl.h): every index of its levels on the host with smaller
list limits, and the sizes of the lists themselves up to 19 strands.  No GPU."""
from __future__ import annotations

import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = ROOT / "tests" / "native" / "glue_scratch_host_check.cpp"
HIPCC = "/opt/rocm/bin/hipcc"


def test_levels_and_list_sizes(tmp_path):
    if not shutil.which(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path / "glue_scratch_host_check"
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-x", "c++", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", str(SRC),
                    "-o", str(out)], check=True, capture_output=True, timeout=600)
    res = subprocess.run([str(out)], capture_output=True, text=True, timeout=600)
    assert res.returncode == 0 and res.stdout.strip().endswith("ALL OK"), res.stdout[-2000:]
