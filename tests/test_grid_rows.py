"""CPU model of the device-wide DP fill (dp_grid_items, RowGrid): one-wave
workers take (pair, strip) items in order from a counter; a strip takes the
values of the row above, 16 columns a block, from 32-bit words that were empty
before the fill and say by themselves that they are there; the worker that
counts a pair's last strip walks its codes.

Modelled, in the kernel's order: the fetch of a block's 16 values a block ahead
(any of them may still be empty), the retry until none is, the stores of a
block's 16 last-row values, each visible at a time of its own, the codes of
every block, which another worker may read only after their writer's release,
the count of done strips and the walk behind it, pairs dropped by their flags,
and the queued pairs that persistent waves take after the grid items.  Every
launch finds its rows empty and its counters at zero.  No schedule may stall, no
value of another fill may be taken, and every pair is walked once, complete."""
import random

import pytest

EMPTY = None


class Fill:
    def __init__(self, pairs, nfill=0, rows=None, drop=(), queue=0, plant="", rng=None):
        self.pairs, self.nfill, self.drop, self.plant, self.rng = pairs, nfill, set(drop), plant, rng
        self.groups = [(Lq + 63) // 64 for Lq, _ in pairs]
        self.items = [(k, s) for k, g in enumerate(self.groups) for s in range(g)]
        if plant == "items not in order":
            self.items.reverse()
        if rows is None or plant != "no refill":
            rows = {(k, s): [EMPTY] * pairs[k][1] for k, s in self.items}
        self.rows = rows
        self.flight = []            # row values stored, not yet visible
        self.codes = {}             # (pair, strip) -> blocks released to the device
        self.done = [0] * len(pairs)
        self.next, self.head = 0, 0
        self.queue = queue
        self.walks, self.queued, self.errors = [], [], []

    def take_value(self, k, s, c, v):
        if v != (self.nfill, k, s, c):
            self.errors.append(f"pair {k} strip {s} column {c}: took {v}")

    def strip(self, k, s):
        Lr = self.pairs[k][1]
        row = self.rows.get((k, s - 1))
        fetch = lambda t: [row[c] for c in range(t, min(t + 16, Lr))]
        nblk, pre = (Lr + 63 + 15) // 16, None

        def above(t, pre):
            while any(v is EMPTY for v in pre) and self.plant != "no retry":
                yield lambda: all(v is not EMPTY for v in fetch(t))
                pre = fetch(t)
            for i, v in enumerate(pre):
                self.take_value(k, s - 1, t + i, v)
            yield None
            return fetch(t + 16)

        if s > 0:
            pre = yield from above(0, fetch(0))
        blocks = 0
        for b in range(nblk):
            t0 = 16 * b
            if s > 0 and t0 + 16 < Lr:
                pre = yield from above(t0 + 16, pre)
            blocks += 1
            if s + 1 < self.groups[k]:
                self.flight += [(k, s, c) for c in range(t0 - 63, t0 - 47) if 0 <= c < Lr]
            yield None
        self.codes[k, s] = blocks                       # release
        yield None
        self.done[k] += 1                               # atomicAdd
        if self.done[k] == self.groups[k] - (self.plant == "walk before the last strip"):
            self.walks.append(k)
            for i in range(self.groups[k]):
                if self.codes.get((k, i)) != nblk:
                    self.errors.append(f"pair {k} walked without the codes of strip {i}")

    def worker(self):
        while self.next < len(self.items):
            k, s = self.items[self.next]
            self.next += 1
            yield None
            if k in self.drop or (self.plant == "a strip dropped" and (k, s) == (0, 0)):
                continue
            yield from self.strip(k, s)
        while self.head < self.queue:
            self.queued.append(self.head)
            self.head += 1
            yield None

    def land(self, n):
        """n of the values in flight become visible, in any order."""
        for _ in range(min(n, len(self.flight))):
            k, s, c = self.flight.pop(self.rng.randrange(len(self.flight)))
            self.rows[k, s][c] = (self.nfill, k, s, c)

    def run(self, nworkers, policy):
        ws = [[self.worker(), None, n] for n in range(nworkers)]
        while ws:
            self.land(self.rng.choice((0, 0, 1, 7, 40)))
            ready = [w for w in ws if w[1] is None or w[1]()]
            if not ready:
                if self.flight:
                    self.land(1)
                    continue
                self.errors.append("stalled")
                return self
            w = self.rng.choice(ready) if policy == "random" else ready[0] if policy == "first" else ready[-1]
            try:
                w[1] = next(w[0])
            except StopIteration:
                ws.remove(w)
        self.land(len(self.flight))
        return self

    def check(self):
        assert not self.errors, self.errors[:3]
        assert sorted(self.walks) == [k for k in range(len(self.pairs)) if k not in self.drop]
        assert self.next == len(self.items) and self.queued == list(range(self.queue))


PAIRS = [(385, 320), (64, 17), (65, 16), (200, 1), (130, 257), (700, 90), (63, 300)]


@pytest.mark.parametrize("nworkers", [1, 2, 5, 64])
@pytest.mark.parametrize("policy", ["random", "first", "last"])
def test_fills_drain(nworkers, policy):
    """Three fills one after another, as launches of one stream: all pairs,
    then some dropped, then persistent waves that go on with queued pairs."""
    rng, rows = random.Random(nworkers), None
    for n, (drop, queue) in enumerate([((), 0), ((0, 4), 0), ((5,), 11)]):
        f = Fill(PAIRS, n, rows, drop, queue, rng=rng).run(nworkers, policy)
        f.check()
        rows = f.rows


@pytest.mark.parametrize("plant", ["no refill", "no retry", "walk before the last strip", "a strip dropped",
                                   "items not in order"])
def test_planted_mistakes_are_seen(plant):
    rng = random.Random(3)
    first = Fill(PAIRS, 0, rng=rng).run(4, "random")
    first.check()
    f = Fill(PAIRS, 1, first.rows, plant=plant, rng=rng).run(2, "random")
    assert f.errors
