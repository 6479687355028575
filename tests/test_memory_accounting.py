"""What a solve holds beside its state: counted by the plan, the jobs and the serving
loop's admission, given up where another buffer needs the room, and left out on request."""
from __future__ import annotations

import pytest

import ofp
import ofp._lib as lib
from ofp import serving

MODS = [4294967291, 4294967279, 4294967231, 65537, 4294967197, 4294967189, 3, 4294967161]
SUMS = 16 * (4 + 8 * 24)  # moduli and sums of up to 16 moduli


def test_sizes():
    def padded(n):
        return sum((x + 63) // 64 * 64 for x in ofp.state_counts(n))
    for n, k in ((3, 1), (12, 3), (14, 8), (20, 5), (22, 14)):
        assert serving.state_bytes(n, k) == padded(n) * k * 4
    assert ofp.extra_bytes(12, 3) == serving.state_bytes(12, 3) + SUMS  # the second pair of arrays
    assert ofp.extra_bytes(16, 8) == SUMS                               # neither pair nor scratch
    assert ofp.extra_bytes(20, 1) == (64 << 20) + SUMS                  # the last step's scratch
    # words of 23, 21 and 19 strands: one array, one per removed arc, one per pair of them
    assert ofp.extra_bytes(22, 14) == (208012 + 22 * 58786 + 231 * 16796) * 14 * 4 + SUMS
    assert ofp.extra_bytes(0, 1) == ofp.extra_bytes(28, 1) == ofp.extra_bytes(12, 0) == 0


class FakeJob:
    """Finishes after a few polls; `room` jobs fit the device, whatever the budget says."""
    live, room, refused = 0, 1, 0

    def __init__(self, ctx, n, moduli):
        if FakeJob.live >= FakeJob.room:
            FakeJob.refused += 1
            raise lib.OfpError(lib.OFP_E_MEMORY, "insufficient HBM")
        FakeJob.live += 1
        self.moduli, self.polls, self.lean = list(moduli), 0, not ctx.extra
        ctx.jobs.append((n, self.lean))

    def enqueue(self, rows):
        pass

    def info(self):
        self.polls += 1
        return type("I", (), {"idle": int(self.polls > 2)})()

    def result(self):
        return [1] * len(self.moduli)

    def close(self):
        FakeJob.live -= 1


class FakeContext:
    def __init__(self):
        self.extra, self.jobs = True, []

    def set_extra_memory(self, on):
        self.extra = on


def _serve(monkeypatch, budget, room, reqs):
    monkeypatch.setattr(serving._lib, "Job", FakeJob)
    FakeJob.live, FakeJob.room, FakeJob.refused = 0, room, 0
    ctx = FakeContext()
    srv = serving.Server(ctx=ctx, budget_bytes=budget, merge=False, tuned=False)
    rep = srv.run([serving.Request(i, n, MODS[:k], 0.0) for i, (n, k) in enumerate(reqs)], poll_s=0.0)
    assert rep["requests"] == len(reqs) and srv.used_bytes == 0 and srv.peak_bytes <= budget
    assert ctx.extra  # as it was
    return ctx.jobs


def test_admission_waits_where_the_device_has_less_than_the_budget(monkeypatch):
    jobs = _serve(monkeypatch, 1 << 40, 1, [(12, 2), (13, 2), (12, 1)])
    assert [n for n, _ in jobs] == [12, 13, 12] and FakeJob.refused > 0
    with pytest.raises(lib.OfpError):  # nothing to wait for
        _serve(monkeypatch, 1 << 40, 0, [(12, 2)])


def test_admission_counts_what_jobs_hold_beside_their_state(monkeypatch):
    one = serving.state_bytes(12, 2) + ofp.extra_bytes(12, 2)
    assert _serve(monkeypatch, 2 * one, 8, [(12, 2), (12, 2)]) == [(12, False)] * 2
    assert FakeJob.refused == 0
    # the state alone fits: alone, with nothing beside it
    assert _serve(monkeypatch, one - 1, 8, [(12, 2), (12, 2)]) == [(12, True)] * 2
    with pytest.raises(RuntimeError):
        _serve(monkeypatch, serving.state_bytes(12, 2) - 1, 8, [(12, 2)])


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(9, 1), (12, 2), (16, 5), (16, 8), (20, 1)])
def test_jobs_hold_what_is_counted(n, k):
    with ofp.Context() as ctx:
        want, _ = ctx.solve(n, MODS[:k])
        for on in (True, False):
            print(f"case job n={n} k={k} extra={on}", flush=True)
            ctx.set_extra_memory(on)
            job = ofp.Job(ctx, n, MODS[:k])
            job.enqueue(n + 1)
            assert job.result() == want
            extra = ofp.extra_bytes(n, k) if on else SUMS
            assert job.info().state_bytes == serving.state_bytes(n, k) + extra
            job.close()
            assert ctx.plan(n, k).state_bytes == serving.state_bytes(n, k)


@pytest.mark.gpu
def test_scratch_gives_way_to_a_larger_state():
    """After a solve that needed scratch, a state fits that fits a fresh context: 48 MB to
    spare, which the lists of 19 strands (17 MB, the context's) leave and the scratch (64 MB) not."""
    m = MODS[:1]
    need = serving.state_bytes(21, 1)
    with ofp.Context() as ctx:
        free = ctx.plan(1, 1).free_bytes
    with ofp.Context(reserve_bytes=free - need - (48 << 20)) as ctx:
        want, _ = ctx.solve(20, m)
        assert ctx.plan(21, 1).fits
        ctx.prepare(21, m)
        got, _ = ctx.solve(20, m)
        assert got == want
