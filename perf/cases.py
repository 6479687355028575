"""The work that programs have this solver do, as cases that can be timed.

Each case is one call sequence through the public entry points of `ofp`: whole
solves of one modulus and of a CRT run's moduli, the solve without device
allocation, a batch of requests through the serving loop, single rows of a
large prepared state, a row's cells on a caller's vectors, and one window of
each half of a row of the multi-GPU layout with the exchange between them.
Sizes are the ones of the CLI, the benchmark, the serving stream and the tests.

A case's inputs are its moduli (primes below 2^32 drawn from the seed, as CRT
runs and requests bring them) and, where the entry point takes vectors, seeded
residues.  All outputs are whole numbers.
"""
from __future__ import annotations

import random
import sys
from pathlib import Path

import numpy as np

PKG = Path(__file__).resolve().parents[1] / "oneesan-gpu_amd"
if str(PKG) not in sys.path:
    sys.path.insert(0, str(PKG))

import ofp  # noqa: E402
from ofp import serving  # noqa: E402

# One context serves all calls of a process, as in the CLI, the CRT runner and a
# service; a second one belongs to the serving loop, which sets launch options.
_ctx = {}


def _context(name: str) -> "ofp.Context":
    if name not in _ctx:
        _ctx[name] = ofp.Context()
    return _ctx[name]


def _is_prime(v: int) -> bool:
    """Miller-Rabin with the bases that decide every v < 4,759,123,141."""
    if v < 2 or any(v % q == 0 for q in (2, 3, 5, 7, 11, 13)):
        return v in (2, 3, 5, 7, 11, 13)
    d, s = v - 1, 0
    while d % 2 == 0:
        d, s = d // 2, s + 1
    for a in (2, 7, 61):
        x = pow(a, d, v)
        if x in (1, v - 1):
            continue
        for _ in range(s - 1):
            x = x * x % v
            if x == v - 1:
                break
        else:
            return False
    return True


def _moduli(rng: random.Random, k: int) -> list[int]:
    """k distinct primes of the 2^20 numbers below 2^32, descending."""
    got: set[int] = set()
    while len(got) < k:
        v = 2**32 - 1 - 2 * rng.randrange(1 << 19)
        if _is_prime(v):
            got.add(v)
    return sorted(got, reverse=True)


def _states(n: int) -> int:
    return sum(ofp.state_counts(n))


def listed() -> list[dict]:
    return [
        # The smallest call: a solve inside a loop that must not allocate.
        {"name": "static_n9_k2", "kind": "static", "n": 9, "k": 2},
        # A small plain solve: launches and host work count.
        {"name": "solve_n12_k1", "kind": "solve", "n": 12, "k": 1},
        # A small solve with an odd number of moduli (the stride is padded).
        {"name": "solve_n15_k3", "kind": "solve", "n": 15, "k": 3},
        # The plain solve of middle size that the benchmark times.
        {"name": "solve_n18_k1", "kind": "solve", "n": 18, "k": 1},
        # Exact runs: every modulus the path bound asks for, in one sweep.
        {"name": "exact_n19_k10", "kind": "solve", "n": 19, "k": 10},
        {"name": "exact_n20_k11", "kind": "solve", "n": 20, "k": 11},
        # A large plain solve: one residue as the CLI is asked for it.
        {"name": "solve_n21_k1", "kind": "solve", "n": 21, "k": 1},
        # Requests that wait together in the serving loop; the two of one n merge.
        {"name": "serve_n14_n16_n17", "kind": "serve", "requests": "14:2,16:8,17:5,16:3"},
        # One full row of a large exact run (13 moduli, stride 14), progress row by row.
        {"name": "row_n21_k13", "kind": "row", "n": 21, "k": 13},
        # One full row with 64-bit ranks (n >= 23), one modulus.
        {"name": "row_n23_k1", "kind": "row", "n": 23, "k": 1},
        # A row's cells on a caller's own vectors, in host memory.
        {"name": "cells_n14_k4", "kind": "cells", "n": 14, "k": 4},
        # The multi-GPU layout: one LOW window's high cells, its exchange into the
        # shares' buckets, and one HIGH window's low cells.
        {"name": "share_n27_k4", "kind": "share", "n": 27, "k": 4, "first": 3, "groups": 8, "high_groups": 4,
         "shares": 8},
    ]


def _cost(n: int, k: int) -> float:
    """A solve's size: states x cells, the index math of a state weighing about
    as much as one and a half moduli."""
    return _states(n) * float((n + 1) * n) * (k + 1.5)


def draw(rng: random.Random) -> dict:
    known = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while (case := _draw(rng)) in known:
        pass
    return case


def _draw(rng: random.Random) -> dict:
    kind = rng.choices(["solve", "static", "serve", "row", "cells", "share"], [10, 2, 3, 3, 2, 2])[0]
    limit = _cost(20, 11)
    if kind == "solve":
        n = rng.randint(9, 21)
        most = max(k for k in range(1, 17) if _cost(n, k) <= limit)
        k = min(most, int(2 ** rng.uniform(0.0, 4.09)))
        return {"kind": "solve", "n": n, "k": k}
    if kind == "static":  # what the static array holds: n = 15 with 8 moduli, n = 16 with 2
        n = rng.randint(7, 16)
        return {"kind": "static", "n": n, "k": rng.randint(1, 2 if n == 16 else 8)}
    if kind == "serve":
        reqs = [(rng.randint(14, 18), rng.randint(1, 8)) for _ in range(rng.randint(2, 5))]
        return {"kind": "serve", "requests": ",".join(f"{n}:{k}" for n, k in reqs)}
    if kind == "row":
        n = rng.randint(18, 23)
        most = max(1, min(16, int(_states(21) * 13 / _states(n))))
        return {"kind": "row", "n": n, "k": rng.randint(1, most)}
    if kind == "cells":
        return {"kind": "cells", "n": rng.randint(8, 14), "k": rng.randint(1, 6)}
    return {"kind": "share", "n": 27, "k": rng.choice([1, 2, 4]), "first": rng.randint(0, 24),
            "groups": rng.randint(2, 8), "high_groups": rng.randint(1, 4), "shares": rng.choice([2, 4, 8])}


def _pairs(case: dict) -> list[tuple[int, int]]:
    return [tuple(int(x) for x in r.split(":")) for r in case["requests"].split(",")]


def prepare(case: dict, seed: int) -> dict:
    rng = random.Random(seed)
    kind = case["kind"]
    state = dict(case)
    if kind in ("solve", "static"):
        state["moduli"] = _moduli(rng, case["k"])
        state["ctx"] = _context("solve")
    elif kind == "serve":
        ctx = _context("serve")
        state["requests"] = [(n, _moduli(rng, k)) for n, k in _pairs(case)]
        state["server"] = serving.Server(ctx, serving.default_budget(ctx))
    elif kind == "row":
        # A state in the middle of a solve: after four rows its words are filled
        # with residues; the timed rows sweep the whole state.
        state["ctx"] = ctx = ofp.Context()
        state["moduli"] = _moduli(rng, case["k"])
        ctx.prepare(case["n"], state["moduli"])
        ctx.row_sweep(4)
        ctx.set_height_caps(False)
        nm, _ = ofp.state_counts(case["n"])
        state["words"] = [i * (nm // 16) for i in range(16)]
    elif kind == "cells":
        state["ctx"] = _context("solve")
        state["moduli"] = mods = _moduli(rng, case["k"])
        nm, nb = ofp.state_counts(case["n"])
        g = np.random.default_rng(seed)
        state["main"] = g.integers(0, mods[-1], (nm, len(mods)), dtype=np.uint32)
        state["blocked"] = np.zeros((nb, len(mods)), np.uint32)
    elif kind == "share":
        state["ctx"] = _context("share")
        state["moduli"] = mods = _moduli(rng, case["k"])
        state["seed"] = rng.randrange(1 << 62)
        info, _, _ = ofp.group_plan(case["n"], case["k"], case["first"], case["high_groups"], high=True)
        g = np.random.default_rng(seed)
        state["main"] = g.integers(0, mods[-1], (info["main_count"], len(mods)), dtype=np.uint32)
    else:
        raise ValueError(f"unknown kind {kind!r}")
    return state


def run(state: dict):
    kind, ctx = state["kind"], state.get("ctx")
    if kind == "solve":
        return ctx.solve(state["n"], state["moduli"])[0]
    if kind == "static":
        return ctx.solve_static(state["n"], state["moduli"])
    if kind == "serve":
        reqs = [serving.Request(i, n, mods, 0.0) for i, (n, mods) in enumerate(state["requests"])]
        state["server"].run(reqs)
        return [r.residues for r in reqs]
    if kind == "row":
        # the state stays on the device; a program reads the words it wants
        ctx.row_sweep(1)
        return np.array([ctx.read_main(i, state["k"]) for i in state["words"]], np.int64)
    if kind == "cells":
        ctx.apply_cells(state["n"], state["moduli"], state["main"], state["blocked"], state["n"], 1, False)
        return {"main": state["main"].view(np.int32), "blocked": state["blocked"].view(np.int32)}
    n, mods, first = state["n"], state["moduli"], state["first"]
    ctx.group_sweep(n, mods, first, state["groups"], seed=state["seed"])
    _, buckets = ctx.group_exchange(n, mods, first, state["groups"], shares=state["shares"], download=True)
    _, main, _ = ctx.group_sweep(n, mods, first, state["high_groups"], seed=state["seed"], high=True,
                                 main_in=state["main"])
    out = {name: a.view(np.int64 if a.dtype == np.uint64 else np.int32) for name, a in buckets.items()}
    out["high_main"] = main.view(np.int32)
    return out


def work(case: dict) -> dict:
    """Bytes: residues read once and written once per row of the grid a solve has
    to sweep.  By the grid's half-turn symmetry half of its rows determine the
    count.  flops: one addition per state, cell and modulus of those rows."""
    kind = case["kind"]

    def solve(n: int, k: int) -> tuple[float, float]:
        rows = (n + 1) / 2
        return 8.0 * k * _states(n) * rows, rows * n * _states(n) * float(k)

    if kind in ("solve", "static"):
        b, f = solve(case["n"], case["k"])
    elif kind == "serve":
        parts = [solve(n, k) for n, k in _pairs(case)]
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    elif kind == "row":
        s = _states(case["n"]) * case["k"]
        b, f = 8.0 * s, float(case["n"]) * s
    elif kind == "cells":
        s = _states(case["n"]) * case["k"]
        b, f = 8.0 * s, float(case["n"]) * s
    else:
        low, _, _ = ofp.group_plan(case["n"], case["k"], case["first"], case["groups"])
        high, _, _ = ofp.group_plan(case["n"], case["k"], case["first"], case["high_groups"], high=True)
        sl, sh = (float(x["main_count"] + x["blocked_count"]) for x in (low, high))
        k = case["k"]
        # the LOW window, its records (8-byte index and residues) and the HIGH window
        b = sl * (8 * k + 8 + 4 * k) + sh * 8 * k
        f = k * (sl * (case["n"] - low["low"]) + sh * high["low"])
    return {"bytes": float(b), "flops": float(f)}


def exact(case: dict, seed: int):
    """Every output is a whole number, compared digit by digit: nothing is rounded."""
    return None
