"""Class tables are packed with the columns the pair kernels load them by
(cell::LdsCols), which need not be those of the height tables: a group sweep's tables
packed by another stride are read out of place on the device.  Checked in the source;
the strides happen to be equal, so no run can tell.  No GPU."""
from __future__ import annotations

import re

from conftest import PKG


def test_group_class_tables_use_the_kernels_columns():
    api = (PKG / "csrc" / "ofp_api.hip").read_text()
    pair = (PKG / "csrc" / "ofp_pair.hip").read_text()
    calls = re.findall(r"pack_(?:group_)?class_table<uint32_t, (\w+)>\(", api)
    assert calls == ["kCols"]
    assert re.search(r"constexpr int kCols = cell::LdsCols<uint32_t>::value;\s*"
                     r"static cell::Pair<uint32_t> t\[kDpRows\]\[kCols\];", api)
    # what the kernels read, and the bytes of one table
    assert pair.count("constexpr int C = LdsCols<Idx>::value;") == 3
    assert len(re.findall(r"load_table<C, C>\(&ctab\[0\]\[0\]", pair)) == 2
    assert "sizeof(Pair<uint32_t>) * LdsCols<uint32_t>::value" in pair
