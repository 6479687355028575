"""Pair passes from one pair of arrays to another (pair_body's Whole in
oneesan-gpu_amd/csrc/ofp_pair_impl.h), built for the host, against the CPU oracle.  No GPU."""
from __future__ import annotations

import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = ROOT / "tests" / "native" / "pair_whole_host_check.cpp"
HIPCC = "/opt/rocm/bin/hipcc"


def test_whole_passes_equal_the_oracle_rows(tmp_path, oracle):
    """n = 2..9: every row of a solve, and whole rows from arbitrary residues, in both
    orders of the classes, at one and three moduli."""
    if not shutil.which(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path / "pair_whole_host_check"
    lib = ROOT / "oracle"
    cmd = [HIPCC, "-O1", "-std=c++17", "-x", "c++", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
           str(SRC), "-o", str(out), f"-L{lib}", "-loracle", f"-Wl,-rpath,{lib}"]
    subprocess.run(cmd, check=True, capture_output=True, timeout=600)
    res = subprocess.run([str(out), "9"], capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stdout[-2000:] + res.stderr[-2000:]
    assert res.stdout.strip().endswith("ALL OK")
    assert res.stdout.count("ok n=") == 64
