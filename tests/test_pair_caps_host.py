"""Height-capped pair passes (oneesan-gpu_amd/csrc/ofp_pair_impl.h), built for the
host: the first rows of a solve against the CPU oracle's whole rows.  No GPU."""
from __future__ import annotations

import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = ROOT / "tests" / "native" / "pair_caps_host_check.cpp"
HIPCC = "/opt/rocm/bin/hipcc"


def test_capped_pairs_equal_the_oracle_rows(tmp_path, oracle):
    """Height-capped pair passes (pair_caps_host_check.cpp): rows 0..W-3 of a solve,
    n = 3..10, each pass over only the classes within its row's height bound."""
    if not shutil.which(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path / "pair_caps_host_check"
    lib = ROOT / "oracle"
    cmd = [HIPCC, "-O1", "-std=c++17", "-x", "c++", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
           str(SRC), "-o", str(out), f"-L{lib}", "-loracle", f"-Wl,-rpath,{lib}"]
    subprocess.run(cmd, check=True, capture_output=True, timeout=600)
    res = subprocess.run([str(out), "10"], capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stdout[-2000:] + res.stderr[-2000:]
    assert res.stdout.strip().endswith("ALL OK")
    assert res.stdout.count("ok n=") == 32
