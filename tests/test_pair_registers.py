"""Registers of the pair kernels in the built library: the passes of the default path
(two workgroups of 256 per CU) keep their values in registers at every moduli count and
both rank widths.  Read from the code objects' own metadata.  No GPU."""
from __future__ import annotations

import re
import shutil
import struct
import subprocess

import pytest

from conftest import PKG

LIB = PKG / "lib" / "libofp.so"
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob: bytes):
    """The device ELF files of a host library's offload bundles."""
    at = blob.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", blob, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(count):
            off, size, tlen = struct.unpack_from("<QQQ", blob, pos)
            triple = blob[pos + 24:pos + 24 + tlen].decode()
            pos += 24 + tlen
            if "gfx950" in triple and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, at + len(MAGIC))


def test_pair_kernels_do_not_spill(tmp_path):
    if not LIB.exists() or not shutil.which(READELF):
        pytest.skip("library or llvm-readelf not available")
    seen = {}
    for i, obj in enumerate(_code_objects(LIB.read_bytes())):
        f = tmp_path / f"{i}.co"
        f.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(f)], check=True, capture_output=True, text=True).stdout
        for name, spill in re.findall(r"\.symbol:\s+(\S+)\.kd.*?\.vgpr_spill_count:\s*(\d+)", notes, re.S):
            seen[name] = int(spill)
    # pair_kernel<KC, Idx, D, GF, MB, Capped>, pair_readers_kernel<KC, Idx, Capped>
    passes = {n: v for n, v in seen.items() if re.search(r"11pair_kernelILi\d+E[jm]Lin?\d+ELi[01]ELi2E", n)}
    readers = {n: v for n, v in seen.items() if "19pair_readers_kernelILi" in n}
    assert len(passes) == 16 * 2 * 5 * 2 and len(readers) == 16 * 2 * 2
    # two at 12 moduli with 64-bit ranks, where the other order is slower
    assert not {n: v for n, v in (passes | readers).items() if v > (2 if "ILi12Em" in n else 0)}


@pytest.mark.gpu
@pytest.mark.parametrize("bits", [0, 64])
@pytest.mark.parametrize("k", [12, 13, 14, 15, 16])
def test_rows_on_both_sides_of_the_change(k, bits, oracle):
    """A row of passes (with and without a launch for all readers) on random vectors at the
    moduli counts around the one from which the sums are gathered first."""
    import numpy as np
    import ofp
    mods = [4294967291, 2, 4294967279, 3, 65537] + [4294967291 - 2 * i for i in range(100, 111)]
    with ofp.Context() as ctx:
        ctx.set_index_width(bits)
        ctx.set_pair_passes(True, 0xFFFFFFFF)
        for n in (4, 12):
            nm, nb = ofp.state_counts(n)
            rng = np.random.default_rng(100 * k + n)
            main = rng.integers(0, 2, (nm, k), dtype=np.uint32) * rng.integers(0, 2**32, (nm, k), dtype=np.uint32)
            main %= np.array(mods[:k], np.uint32)
            blk = np.zeros((nb, k), np.uint32)
            got = main.copy()
            print(f"case row n={n} k={k} bits={bits}", flush=True)
            ctx.apply_cells(n, mods[:k], got, blk, n, 1, False)
            for j, m in enumerate(mods[:k]):
                want, b = np.ascontiguousarray(main[:, j]), np.zeros(nb, np.uint32)
                oracle.apply_cells(n, m, want, b, n, 1, False)
                assert np.array_equal(got[:, j], want), (n, k, j)
