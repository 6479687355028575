"""Who chooses how two cells run: the library by size, unless a table entry of the very
same (n, k), timed against that choice on whole solves, was faster -- through the tuner,
the serving loop and the C ABI's way back to the library's choice."""
from __future__ import annotations

import pytest


class Recorder:
    """A context that only remembers its settings."""

    def __init__(self):
        self.set = {}

    def __getattr__(self, name):
        if not name.startswith("set_"):
            raise AttributeError(name)
        return lambda *a: self.set.__setitem__(name[4:], a)


def _applied(n, k):
    from ofp import autotune
    ctx = Recorder()
    autotune.apply(ctx, n, k)
    return ctx.set["pair_passes"]


def test_apply_leaves_the_choice_to_the_library(tmp_path, monkeypatch):
    from ofp import autotune
    packaged = autotune.load_cache(autotune.PACKAGED)
    for n in range(1, 28):
        for k in range(1, 17):
            ent = packaged.get(f"n={n},k={k}", {})
            if ent.get("pair_choice") != "table":
                assert _applied(n, k) == (-1, 0), (n, k)
    # an entry without a timed choice (an older table's) says nothing; one of the same n but
    # other moduli neither
    table = tmp_path / "pk.json"
    ent = {"threads": 256, "blocks_per_cu": 32, "pair_mode": 1, "pair_mask": 0x10000}
    autotune.save_cache({"n=16,k=8": ent, "n=17,k=8": dict(ent, pair_choice="table"),
                         "n=18,k=8": dict(ent, pair_choice="library")}, table)
    monkeypatch.setattr(autotune, "PACKAGED", table)
    assert _applied(16, 8) == (-1, 0)
    assert _applied(17, 8) == (1, 0x10000)
    assert _applied(17, 11) == (-1, 0)
    assert _applied(18, 8) == (-1, 0)


def test_tables_settings_stand_only_where_faster(monkeypatch):
    from ofp import autotune
    ent = {"layout": 1, "threads": 128, "blocks_per_cu": 8, "cap_percent": 95, "pair_mode": 1, "pair_mask": 0x550}

    def chosen(own, tuned, table):
        ctx = Recorder()
        ms = {(256, -1): own, (128, -1): tuned, (128, 1): table}
        monkeypatch.setattr(autotune, "solve_ms",
                            lambda c, n, m: ms[c.set["launch"][0], c.set["pair_passes"][0]])
        e = autotune.choose_stage(ctx, 16, [3, 5], ent)
        assert e["solve_ms"] == ms[ctx.set["launch"][0], ctx.set["pair_passes"][0]]
        assert e["threads"] == ctx.set["launch"][0] and e["cap_percent"] in autotune.CAP_PERCENTS
        return e["threads"], e["pair_choice"]
    assert chosen(1.0, 0.99, 0.985) == (256, "library")  # no faster than runs differ
    assert chosen(1.0, 0.9, 0.89) == (128, "library")
    assert chosen(1.0, 1.2, 0.8) == (128, "table")


def test_packaged_entries_are_timed_choices():
    from ofp import autotune
    for key, ent in autotune.load_cache(autotune.PACKAGED).items():
        k = int(key.split(",")[1][2:])
        assert ent.get("pair_choice") in ("library", "table") and ent["solve_ms"] > 0, key
        # a split that is none at k moduli would split the larger counts that fall back to it
        assert ent["low_cells"] == 0 or ent["low_kc"] < k, key


MODS = [4294967291, 4294967279, 65537]


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(9, 2), (12, 1), (16, 3), (18, 2)])
def test_tuned_and_served_contexts_run_the_librarys_passes(n, k):
    """The launches of a solve are those of a fresh context after the tuner's settings,
    after serving, and after passes were switched on and the choice given back."""
    import ofp
    from ofp import autotune, serving
    mods = MODS[:k]
    with ofp.Context() as ctx:
        want, st = ctx.solve(n, mods)
    fresh = st["launches"]
    with ofp.Context() as ctx:
        ctx.set_pair_passes(0)
        assert ctx.solve(n, mods)[1]["launches"] != fresh
        ctx.set_pair_passes(-1)
        got, st = ctx.solve(n, mods)
        assert got == want and st["launches"] == fresh
    if not any(e.get("pair_choice") == "table" for key, e in autotune.load_cache(autotune.PACKAGED).items()
               if key == f"n={n},k={k}"):
        with ofp.Context() as ctx:
            autotune.apply(ctx, n, k)
            ctx.set_height_caps(True)
            assert ctx.solve(n, mods)[1]["launches"] == fresh
    with ofp.Context() as ctx:
        reqs = [serving.Request(0, 10, MODS, 0.0), serving.Request(1, 16, MODS[:2], 0.0)]
        serving.Server(ctx, serving.default_budget(ctx)).run(reqs)
        for set_, v in ((ctx.set_layout, (1,)), (ctx.set_launch, (0, 0)), (ctx.set_variant, (2,)), (ctx.set_low_cells, (0, 16)),
                        (ctx.set_height_caps, (True,)), (ctx.set_xcd_pieces, (5,)), (ctx.set_sorted_cells, (-1,))):
            set_(*v)
        assert ctx.solve(n, mods)[1]["launches"] == fresh


@pytest.mark.gpu
def test_choice_changed_in_the_middle_of_a_solve(oracle):
    """Rows under the library's choice, one launch per cell and passes in place, in turn on
    one state (the second pair of arrays keeps an older state meanwhile)."""
    import ofp
    n, mods = 11, MODS
    want = [oracle.solve(n, m) for m in mods]
    with ofp.Context() as ctx:
        for modes in ((-1, 0, 1), (0, -1, -1, 1), (1, 1, -1, 0, 0)):
            ctx.set_pair_passes(-1)
            ctx.prepare(n, mods)
            for r in range(n + 1):
                ctx.set_pair_passes(modes[r % len(modes)])
                ctx.row_sweep(1)
            assert ctx.read_main(0, len(mods)) == want, modes
