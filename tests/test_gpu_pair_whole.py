"""Small states' pair passes (one launch to a second pair of arrays, the default below a
state size) against cells launched one by one, through the C ABI, bit-exact."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu

MODS = [4294967291, 2, 4294967279, 65537, 4294967197, 3, 4294967161, 4294967143, 4294967111]


@pytest.fixture(scope="module")
def cells_ctx():
    import ofp
    ctx = ofp.Context()
    ctx.set_pair_passes(False)
    yield ctx
    ctx.close()


@pytest.fixture()
def small_ctx():
    import ofp
    ctx = ofp.Context()
    yield ctx
    ctx.close()


def _words(ctx, n, k):
    import ofp
    count = ofp.state_counts(n)[0]
    return [ctx.read_main(i, k) for i in sorted({0, 1, 2, count // 3, count // 2, count - 2, count - 1} & set(range(count)))]


@pytest.mark.parametrize("n,k", [(2, 1), (2, 8), (3, 1), (4, 3), (5, 8), (6, 2), (9, 1), (9, 9), (11, 7), (12, 8), (14, 5),
                                 (15, 8), (16, 5), (16, 6), (17, 2), (17, 3)])
def test_rows_and_solves(small_ctx, cells_ctx, n, k):
    """Odd and even rows, every moduli count of a launch and one more, both sides of the
    size limit: rows one by one and together, a state reused and one that grows."""
    print(f"case small passes n={n} k={k}", flush=True)
    mods = MODS[:k]
    want = cells_ctx.solve(n, mods)[0]
    assert small_ctx.solve(n, mods)[0] == want
    for caps in (True, False):
        for rows in (1, n // 2, n + 1):
            got = []
            for ctx in (small_ctx, cells_ctx):
                ctx.set_height_caps(caps and rows == n + 1)
                ctx.prepare(n, mods)
                ctx.row_sweep(rows - 1)
                ctx.row_sweep(1)
                got.append(_words(ctx, n, k) if rows <= n else ctx.read_main(0, k))
                ctx.set_height_caps(True)
            assert got[0] == got[1], (caps, rows)
    assert small_ctx.solve(n, mods)[0] == want
    if k <= 8 and n <= 12:
        assert small_ctx.solve_static(n, mods) == want


def test_settings_changed_between_rows(small_ctx, cells_ctx):
    """A state prepared under one setting and swept under another, in both directions."""
    n, mods = 13, MODS[:3]
    want = cells_ctx.solve(n, mods)[0]
    for first, then in ((64, 0), (0, 64)):
        small_ctx.solve(n, mods)  # the second pair of arrays holds an old state
        small_ctx.set_index_width(first)
        small_ctx.prepare(n, mods)
        small_ctx.row_sweep(5)
        small_ctx.set_index_width(then)
        small_ctx.row_sweep(n + 1 - 5)
        assert small_ctx.read_main(0, 3) == want
        small_ctx.set_index_width(0)
    small_ctx.prepare(n, mods)
    small_ctx.row_sweep(3)
    small_ctx.set_pair_passes(True)
    small_ctx.row_sweep(4)
    small_ctx.set_pair_passes(False)
    small_ctx.row_sweep(n + 1 - 7)
    assert small_ctx.read_main(0, 3) == want
