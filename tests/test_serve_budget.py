"""Admission of the serving loop (no GPU): the scenarios' memory and the room
the batch's increments are given stay within the budget, and a request that
fits the budget alone is served."""
import pytest

from magic_master_amd import hip, serve


class FakeBatch:
    """Every scenario ends after three runs."""

    def __init__(self, *a, **k):
        FakeBatch.one = self
        self.room, self.left, self.grids, self.seen = 0, {}, {}, []

    def set_increment_room(self, nbytes):
        assert nbytes >= 1
        self.room = nbytes

    def add(self, g, *a):
        s = next(k for k in range(1000) if k not in self.left)
        self.left[s], self.grids[s] = 3, g
        return s

    def start(self, s, t, tend, *a):
        self.tend = tend

    def run(self, **k):
        self.seen.append((sum(serve.footprint_bytes(g) for g in self.grids.values()) + self.room, self.room, len(self.grids)))
        for s in self.left:
            self.left[s] -= 1

    def state(self, s):
        return {"status": 0, "active": self.left[s] > 0, "nsteps": 3, "rejects": 0, "t": 1e9, "dt": 1.0}

    def remove(self, s):
        del self.left[s], self.grids[s]

    def global_sums(self, s):
        return [0.0] * 6

    def close(self):
        pass


@pytest.mark.parametrize("share", [1.01, 1.1, 2.5, 6.0])   # of the largest request's own memory
def test_increments_count_against_the_budget(monkeypatch, share):
    monkeypatch.setattr(hip, "MagicBatch", FakeBatch)
    rq = serve.poisson_requests(100.0, 0.2, seed=3, nmin=(64, 64, 96), nmax=(200, 200, 300))
    assert len(rq) >= 10
    for r in rq:
        r.arrival = 0.0
    budget = share * max(serve.footprint_bytes(r.grid) for r in rq)
    res = serve.Server(budget_bytes=budget, snapshots="none").run(rq)
    assert all(o.status == 0 and o.steps == 3 for o in res["outcomes"])
    seen = FakeBatch.one.seen
    assert max(total for total, _, _ in seen) <= budget
    assert res["max_footprint_bytes"] == max(total for total, _, _ in seen)
    full = serve.increment_room(budget, [r.grid for r in rq])
    assert all(room == full for _, room, n in seen if n > 1)
    assert max(n for _, _, n in seen) >= (2 if share > 2 else 1)
