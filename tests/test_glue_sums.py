"""The 64-bit sums of a half-row solve's last step (class_shape in
oneesan-gpu_amd/csrc/ofp_glue_impl.h) stay below 2^64 at every width, moduli count and
CU count, checked on the host with the kernel's walk over its tasks.  No GPU."""
from __future__ import annotations

import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = ROOT / "tests" / "native" / "glue_sums_host_check.cpp"
HIPCC = "/opt/rocm/bin/hipcc"


def test_no_sum_can_wrap(tmp_path):
    if not shutil.which(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path / "glue_sums_host_check"
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-x", "c++", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", str(SRC),
                    "-o", str(out)], check=True, capture_output=True, timeout=600)
    res = subprocess.run([str(out)], capture_output=True, text=True, timeout=600)
    assert res.returncode == 0 and res.stdout.strip().endswith("ALL OK"), res.stdout[-2000:]
