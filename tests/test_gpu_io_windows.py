"""Windows of group sweeps and the exchange's buckets with an odd moduli count, whose
records are padded on the device: callers' arrays go through the copy buffer in pieces
(64 MiB, several per array here), against the same words with an even count, which are
copied at once."""
from __future__ import annotations

import numpy as np
import pytest

import ofp
from ofp.path_bound import PRIMES

pytestmark = pytest.mark.gpu


def test_odd_windows_in_pieces():
    n, low, groups = 17, 6, 64
    mods = PRIMES[:6]
    rng = np.random.default_rng(17)
    info, _, _ = ofp.group_plan(n, 6, 0, groups, low=low)
    assert info["main_count"] * 20 > 2 * (64 << 20) and info["blocked_count"] * 20 > 64 << 20
    main = rng.integers(0, mods[-1], (info["main_count"], 6), dtype=np.uint32)
    got = {}
    with ofp.Context() as ctx:
        for k in (6, 5):
            print(f"case low window k={k}", flush=True)
            _, m, b = ctx.group_sweep(n, mods[:k], 0, groups, low, main_in=main[:, :k], blocked_out=True)
            print(f"case exchange k={k}", flush=True)
            _, x = ctx.group_exchange(n, mods[:k], 0, groups, low, shares=4, download=True)
            high, _, _ = ofp.group_plan(n, k, 0, 1 << (n - low), low=low, high=True)
            print(f"case high window k={k}", flush=True)
            _, h, _ = ctx.group_sweep(n, mods[:k], 0, 1 << (n - low), low, main_in=main[:high["main_count"], :k], high=True,
                                      blocked_in=np.resize(b, (high["blocked_count"], k)))
            got[k] = (m, b, x["main_res"], x["blocked_res"], h)
            if k == 6:
                index = (x["main_index"], x["blocked_index"])
    assert np.array_equal(index[0], x["main_index"]) and np.array_equal(index[1], x["blocked_index"])
    for a, b in zip(got[6], got[5]):
        assert a.shape[0] == b.shape[0] and np.array_equal(a[:, :5], b)
