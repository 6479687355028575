"""The kernels load only the columns of their height tables that a row of width W can
read (used_cols in oneesan-gpu_amd/csrc/ofp_cell_impl.h: (W+1)/2 + 3): no word of W
positions is higher than (W+1)/2 where it can still be completed, and the scans read
two heights above a word's own.  Checked with the oracle's height DP."""
from __future__ import annotations

import re

from conftest import PKG


def test_heights_fit_the_loaded_columns(oracle):
    lib = oracle.load()
    text = (PKG / "csrc" / "ofp_cell_impl.h").read_text()
    assert re.search(r"used_cols\(int W\) \{ return \(W \+ 1\) / 2 \+ 3; \}", text)
    for W in range(2, 29):
        top = max(h for j in range(W + 1) for h in range(32) if h <= 1 + j and lib.or_dp(W - j, h) > 0)
        assert top <= (W + 1) // 2, W
        assert top + 2 < (W + 1) // 2 + 3 <= 22, W  # within the LDS columns of both widths
