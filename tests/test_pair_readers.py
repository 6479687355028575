"""The readers of a pair pass in one launch (pair_readers_kernel in
oneesan-gpu_amd/csrc/ofp_pair.hip): its pieces on the host, and its solves and rows on
the GPU against the CPU oracle."""
from __future__ import annotations

import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = ROOT / "tests" / "native" / "pair_readers_host_check.cpp"
HIPCC = "/opt/rocm/bin/hipcc"
MODS = [4294967291, 4294967279, 65537, 2, 4294967231, 3, 4294967197, 4294967189, 4294967161]


def test_pieces_hold_every_class_once(tmp_path):
    if not shutil.which(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path / "pair_readers_host_check"
    subprocess.run([HIPCC, "-O1", "-std=c++17", "-x", "c++", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", str(SRC),
                    "-o", str(out)], check=True, capture_output=True, timeout=600)
    res = subprocess.run([str(out)], capture_output=True, text=True, timeout=600)
    assert res.returncode == 0 and res.stdout.strip().endswith("ALL OK"), res.stdout[-2000:]


@pytest.mark.gpu
@pytest.mark.parametrize("bits", [0, 64])
@pytest.mark.parametrize("n, k", [(3, 1), (4, 2), (7, 9), (10, 1), (10, 3), (12, 1), (12, 9), (13, 2)])
def test_every_cell_paired(bits, n, k, oracle):
    """Pair passes at every pair of cells (sizes from below one piece to many pieces of a
    chunk, capped rows and whole ones): residues equal the oracle's."""
    import ofp
    with ofp.Context() as ctx:
        ctx.set_index_width(bits)
        ctx.set_pair_passes(True, 0xFFFFFFFF)
        assert ctx.solve(n, MODS[:k])[0] == [oracle.solve(n, m) for m in MODS[:k]]
        ctx.set_height_caps(False)  # all rows, whole
        assert ctx.solve(n, MODS[:k])[0] == [oracle.solve(n, m) for m in MODS[:k]]


@pytest.mark.gpu
def test_second_pair_of_arrays_has_the_small_states_size(oracle):
    """A small solve on a context that holds a large state takes a second pair of arrays of
    its own size, and the large state's arrays serve the next large solve."""
    import ofp
    with ofp.Context() as ctx, ofp.Context() as other:  # the other one holds no state
        big = ctx.solve(18, MODS[:8])[0]
        free = other.plan(12, 1).free_bytes
        for n in (12, 11, 12):
            assert ctx.solve(n, MODS[:1])[0] == [oracle.solve(n, MODS[0])]
        assert free - other.plan(12, 1).free_bytes < 64 << 20
        assert ctx.solve(18, MODS[:8])[0] == big
