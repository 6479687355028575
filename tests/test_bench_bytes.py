"""Declared bytes of a solve's height-capped rows in the benchmark: a pass over two cells
counts once.  No GPU."""
from __future__ import annotations

import sys

from conftest import ROOT

sys.path.insert(0, str(ROOT))


def test_passes_count_once():
    import bench
    import ofp
    n, k, pct = 19, 3, 85
    W = n + 1
    nm, nb = ofp.state_counts(n)
    rows = [r for r in range(W) if any(ofp.height_cap(n, r, p, pct)[0] for p in range(1, W))]
    assert rows

    def words(r, p):
        cap, blk = ofp.height_cap(n, r, p, pct)
        return blk + bench.capped_words(W, cap) if cap else nm + nb
    single = sum(8.0 * k * words(r, p) for r in rows for p in range(1, W))
    assert bench.capped_rows_bytes(n, k, pct, set()) == single
    pairs = set(range(W - 1, 1, -2))
    got = bench.capped_rows_bytes(n, k, pct, pairs)
    # every pair of cells at once where it is large, at no less than the greater of the two
    low = sum(8.0 * k * max(words(r, p), words(r, p - 1)) for r in rows for p in range(W - 1, 1, -2))
    assert low <= got < 0.75 * single


def test_rate_of_a_large_solve_is_possible():
    """n=22 at 14 moduli: 2.69 s of capped rows as measured stay below the HBM peak."""
    import bench
    got = bench.capped_rows_bytes(22, 14, 85, set(range(22, 1, -2)))
    assert got / 2.69 / 1e9 < bench.HBM_PEAK_GBS
