"""CPU model of the row handoff between the waves of one workgroup
(k_dp_mw, RowLds): the waits, reads, writes and progress words of every
block of 16 steps in their order, under schedules that interleave the waves
at every wait.  No schedule may deadlock, and every value read must be the one
that the strip above stored for that column."""
import random

import pytest

RING = 256


def wave(m, w):
    """Generator of wave w: yields (kind, wave, need) before a wait."""
    W, Lr, ns = m.W, m.Lr, m.ns
    for s in range(w, ns, W):
        for t0 in range(0, Lr + 63, 16):
            if s > 0 and t0 < Lr:
                above = (w - 1) % W
                if w == 0:
                    if t0 % 64 == 0:
                        yield m.stored, above, ((s - 1) << 16) | min(t0 + 64, Lr)
                        for c in range(t0, min(t0 + 64, Lr)):
                            m.check(m.row.get(c), s - 1, c)
                else:
                    cols = min(t0 + 16, Lr)
                    yield m.stored, above, ((s - 1) << 16) | cols
                    for c in range(t0, cols):
                        m.check(m.ring[above].get(c % RING), s - 1, c)
                    m.taken[w] = (s << 16) | cols
            cols = t0 - 47
            if s + 1 == ns or cols <= 0:
                continue
            mine = [c for c in range(t0 - 63, t0 - 47) if 0 <= c < Lr]
            if w == W - 1:
                for c in mine:
                    m.row[c] = (s, c)
                if cols % 64 < 16 or cols >= Lr:
                    m.stored[w] = (s << 16) | min(cols, Lr)
                continue
            cols = min(cols, Lr)
            need = (((s + 1) << 16) | (cols - RING) if cols > RING else
                    ((s - W + 1) << 16) | Lr if s >= W else 0)
            if need and not m.free:
                yield m.taken, w + 1, need
            for c in mine:
                m.ring[w][c % RING] = (s, c)
            m.stored[w] = (s << 16) | cols


class Model:
    def __init__(self, W, ns, Lr, free=False):
        self.W, self.ns, self.Lr, self.free = W, ns, Lr, free
        self.stored, self.taken = [0] * W, [0] * W
        self.ring, self.row = [{} for _ in range(W)], {}
        self.wrong = 0

    def check(self, got, s, c):
        self.wrong += got != (s, c)

    def run(self, policy, rng):
        waves = {w: wave(self, w) for w in range(self.W)}
        wait = {w: None for w in waves}
        while waves:
            ready = [w for w in waves if wait[w] is None or wait[w][0][wait[w][1]] >= wait[w][2]]
            if not ready:
                return False
            w = rng.choice(ready) if policy == "random" else min(ready) if policy == "writers" else max(ready)
            try:
                wait[w] = next(waves[w])
            except StopIteration:
                del waves[w]
        return True


@pytest.mark.parametrize("W", [4, 8, 16])
@pytest.mark.parametrize("ns,Lr", [(2, 17), (5, 1), (11, 300), (11, 1500), (16, 64), (17, 255), (37, 257), (40, 900)])
def test_mw_handoff(W, ns, Lr):
    for policy in ("random", "writers", "readers"):
        m = Model(W, ns, Lr)
        assert m.run(policy, random.Random(W * 1000 + ns)), "deadlock"
        assert m.wrong == 0


def test_mw_handoff_model_sees_a_missing_wait():
    # without the wait for the strip below, a writer runs over its ring
    m = Model(4, 4, 900, free=True)
    m.run("writers", random.Random(1))
    assert m.wrong > 0
