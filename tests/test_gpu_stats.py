"""What ofp_stats counts: the cells a call applied (half of a solve's where it runs from
half of its rows), the rows it advanced, and its launches."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu

MODS = [4294967291, 4294967279, 65537]


@pytest.mark.parametrize("n,k", [(2, 1), (3, 2), (8, 3), (9, 1), (16, 2)])
def test_transitions_are_those_performed(gpu_ctx, n, k):
    import ofp
    mods, W = MODS[:k], n + 1
    cell = sum(ofp.state_counts(n)) * k
    print(f"case stats n={n} k={k}", flush=True)
    half = W >= 4  # narrower solves run all their rows
    st = gpu_ctx.solve(n, mods)[1]
    assert st["rows"] == W and st["transitions"] == W * (W - 1) // (2 if half else 1) * cell
    gpu_ctx.set_height_caps(False)
    try:
        st = gpu_ctx.solve(n, mods)[1]
        assert st["rows"] == W and st["transitions"] == W * (W - 1) * cell
    finally:
        gpu_ctx.set_height_caps(True)
    gpu_ctx.prepare(n, mods)
    st = gpu_ctx.row_sweep(2)
    assert st["rows"] == 2 and st["transitions"] == 2 * (W - 1) * cell


def test_sweeps_add_up(gpu_ctx):
    import ofp
    n, W = 10, 11
    gpu_ctx.set_max_batch(1)
    try:
        st = gpu_ctx.solve(n, MODS)[1]
    finally:
        gpu_ctx.set_max_batch(0)
    assert st["rows"] == 3 * W and st["transitions"] == 3 * W * (W - 1) // 2 * sum(ofp.state_counts(n))
