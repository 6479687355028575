"""Callers' vectors whose stride differs from the device's go through a copy buffer in
pieces: more states than one piece holds (64 MiB), odd moduli counts and both layouts,
against the same cells with an even count (copied at once)."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MODS = [4294967291, 4294967279, 4294967231, 4294967197]


@pytest.mark.parametrize("layout", [1, 0])
@pytest.mark.parametrize("n,cells", [(17, (9, 9)), (6, (6, 5))])
def test_vectors_in_pieces(n, cells, layout):
    import ofp
    nm, nb = ofp.state_counts(n)
    rng = np.random.default_rng(7)
    main = rng.integers(0, MODS[-1], (nm, 4), dtype=np.uint32)
    blk = rng.integers(0, MODS[-1], (nb, 4), dtype=np.uint32)
    with ofp.Context(layout=1) as ctx:
        m4, b4 = main.copy(), blk.copy()
        ctx.apply_cells(n, MODS, m4, b4, *cells, True)
    with ofp.Context(layout=layout) as ctx:
        for k in (3, 1):
            print(f"case pieces n={n} k={k} layout={layout}", flush=True)
            m, b = np.ascontiguousarray(main[:, :k]), np.ascontiguousarray(blk[:, :k])
            ctx.apply_cells(n, MODS[:k], m, b, *cells, True)
            assert np.array_equal(m, m4[:, :k]) and np.array_equal(b, b4[:, :k])
