"""Solves from half of their rows (height caps on: only the answer word is read)
against solves that sweep every row (caps off), through the C ABI, bit-exact."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu

MODS = [4294967291, 2, 4294967279, 4294967231, 65537, 4294967197, 4294967189, 3, 4294967161, 4294967143, 4294967111,
        4294967087, 4294967029, 4294966997, 4294966981, 4294966943, 4294966927]


def _whole(ctx, n, mods):
    ctx.set_height_caps(False)
    try:
        return ctx.solve(n, mods)[0]
    finally:
        ctx.set_height_caps(True)


@pytest.mark.parametrize("bits", [0, 64])
@pytest.mark.parametrize("n,ks", [(3, (1, 2)), (4, (3,)), (7, (1, 17)), (10, (2, 5)), (11, (6,)), (12, (1, 3)), (14, (4, 17)),
                                  (15, (1,)), (16, (1, 2, 6)), (17, (3,)), (18, (1, 5)), (20, (1, 3))])
def test_half_rows_equal_whole_solves(gpu_ctx, n, ks, bits):
    """Widths on both sides of every change of the last step: odd and even W, 11, 13,
    17, 19 and 21 strands, one to five moduli passes, padded strides, both rank widths."""
    try:
        gpu_ctx.set_index_width(bits)
        for k in ks:
            print(f"case half rows n={n} k={k} bits={bits}", flush=True)
            mods = MODS[:k]
            got, st = gpu_ctx.solve(n, mods)
            assert got == _whole(gpu_ctx, n, mods), (n, k)
            assert gpu_ctx.read_main(0, k) is not None and st["rows"] == n + 1
            gpu_ctx.solve(n, mods)
            assert gpu_ctx.read_main(0, k) == got  # the answer word holds the residues
    finally:
        gpu_ctx.set_index_width(0)


def test_jobs_and_static_solves(gpu_ctx):
    """Jobs side by side (all rows at once: half of them; rows one by one: all of
    them) and the static solve give the residues of whole solves."""
    import ofp
    sizes = [(14, 3), (15, 2), (16, 1), (13, 5)]
    want = [_whole(gpu_ctx, n, MODS[:k]) for n, k in sizes]
    jobs = [ofp.Job(gpu_ctx, n, MODS[:k]) for n, k in sizes]
    for j, (n, _) in zip(jobs[:3], sizes):
        j.enqueue(n + 1)
    for _ in range(sizes[3][0] + 1):
        jobs[3].enqueue(1)
    print("case jobs", flush=True)
    assert [j.result() for j in jobs] == want
    for j in jobs:
        j.close()
    for (n, k), w in zip(sizes, want):
        print(f"case static n={n} k={k}", flush=True)
        assert gpu_ctx.solve_static(n, MODS[:k]) == w
