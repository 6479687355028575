"""The half-row solve's last step (oneesan-gpu_amd/csrc/ofp_glue_impl.h), built for
the host: the lists of open meanders against a walk along the arcs of every pair of
words (up to 13 strands), and whole solves n = 3..11 -- the oracle sweeps half of
the cells, the header's functions sum over the meeting pairs -- against the oracle's
whole solves for three moduli including 2.  No GPU."""
from __future__ import annotations

import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = ROOT / "tests" / "native" / "glue_host_check.cpp"
HIPCC = "/opt/rocm/bin/hipcc"


def test_half_of_the_rows_give_the_whole_count(tmp_path, oracle):
    if not shutil.which(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path / "glue_host_check"
    lib = ROOT / "oracle"
    cmd = [HIPCC, "-O1", "-std=c++17", "-x", "c++", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
           str(SRC), "-o", str(out), f"-L{lib}", "-loracle", f"-Wl,-rpath,{lib}"]
    subprocess.run(cmd, check=True, capture_output=True, timeout=600)
    res = subprocess.run([str(out), "11"], capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stdout[-2000:] + res.stderr[-2000:]
    assert res.stdout.strip().endswith("ALL OK")
    assert res.stdout.count("\nok n=") == 27
