"""CPU: the hand-off of the bulge chasing between waves (chase in wantibexos_amd/csrc/k_band.hip),
as a model whose steps are interleaved at random.

A workgroup takes SW sweeps at a time, one wave each, and one wave more that loads what the
sweep before the group left.  Boundary i (what sweep i of the group reads) is a ring of R
slots with a count of tasks written and one of tasks read; between groups a count of finished
tasks in memory.  Checked: every task finds in its two slots the tasks k and k + 1 of the sweep
before, a slot is not written while its reader needs it, the tasks of sweep s - 1 up to k + 1
are done before task k of sweep s, and every wave ends; when waits give up (a limit of a few
polls) every wave still ends, and if anything is left undone the error flag is set."""
import random

import pytest


def ntasks(N, b, s):
    return 1 + (N - 2 - s) // b


class Group:
    def __init__(self, SW, R):
        self.wrote, self.read = [0] * SW, [0] * SW
        self.slot = [[None] * R for _ in range(SW)]
        self.bad, self.group = False, None
        self.at_barrier, self.left_at = 0, []     # arrivals; where waves left


class Model:
    def __init__(self, N, b, SW, R, nwg, limit=None, ahead=2, room=0, check_bad=True):
        self.N, self.b, self.SW, self.R, self.nwg, self.limit = N, b, SW, R, nwg, limit
        self.ahead, self.room, self.check_bad = ahead, room, check_bad
        self.err, self.claim = False, 0
        self.prog = [0] * (N // SW + 2)
        self.done = {s: 0 for s in range(-1, N)}
        self.done[-1] = ntasks(N, b, -1)
        self.waves = [self.wave(w, g) for g in (Group(SW, R) for _ in range(nwg)) for w in range(SW + 1)]

    def give_up(self, g):
        g.bad = self.err = True

    def wait(self, g, count, need, memory=False):
        """a generator: True once count() >= need, False when given up"""
        n = 0
        while count() < need:
            if g.bad and not memory:
                return False
            if (memory and self.err) or (self.limit is not None and n > self.limit):
                self.give_up(g)
                return False
            n += 1
            yield
        return True

    def missing(self, g, phase):
        """arrivals at the barriers so far that waves which have left do not make"""
        return sum(max(0, phase - p) for p in g.left_at)

    def wave(self, w, g):
        N, b, SW, R = self.N, self.b, self.SW, self.R
        phase = 0
        loaded = 0
        while True:
            phase += 1
            g.at_barrier += 1
            while g.at_barrier < phase * (SW + 1) - self.missing(g, phase):
                yield
            yield
            if self.check_bad and g.bad:
                g.left_at.append(phase)
                return
            if w == 0:
                g.group, self.claim = self.claim, self.claim + 1
                g.wrote, g.read = [0] * SW, [0] * SW
            phase += 1
            g.at_barrier += 1
            while g.at_barrier < phase * (SW + 1) - self.missing(g, phase):
                yield
            yield
            gi = g.group
            s0 = gi * SW
            if s0 > N - 2:
                g.left_at.append(phase)
                return
            if w == SW:
                ntp = ntasks(N, b, s0 - 1)
                for k in range(ntp):
                    if gi > 0:
                        if not (yield from self.wait(g, lambda: self.prog[gi - 1], k + 1, memory=True)):
                            g.left_at.append(phase)
                            return
                    if not (yield from self.wait(g, lambda: g.read[0], k + 1 - R - self.room)):
                        g.left_at.append(phase)
                        return
                    assert gi == 0 or self.done[s0 - 1] >= k + 1
                    g.slot[0][k % R] = (s0 - 1, k)
                    yield
                    g.wrote[0] = k + 1
                    loaded += 1
                    assert loaded < 4 * N * N, "the loader goes round"
                continue
            s = s0 + w
            if s > N - 2:
                continue
            last = w == SW - 1 or s == N - 2
            nt, ntp = ntasks(N, b, s), ntasks(N, b, s - 1)
            for k in range(nt):
                if not (yield from self.wait(g, lambda: g.wrote[w], min(k + self.ahead, ntp))):
                    g.left_at.append(phase)
                    return
                assert g.slot[w][k % R] == (s - 1, k)
                yield
                if k + 1 < ntp:
                    assert g.slot[w][(k + 1) % R] == (s - 1, k + 1)
                g.read[w] = k + 1
                yield
                if last:
                    self.done[s] = k + 1
                    if k > 0:
                        self.prog[gi] = k             # task k - 1's stores are complete
                else:
                    if not (yield from self.wait(g, lambda: g.read[w + 1], k + 1 - R - self.room)):
                        g.left_at.append(phase)
                        return
                    g.slot[w + 1][k % R] = (s, k)
                    yield
                    g.wrote[w + 1] = k + 1
                    self.done[s] = k + 1
            if last:
                self.prog[gi] = nt

    def run(self, rng, steps=4_000_000):
        live = list(self.waves)
        while live:
            steps -= 1
            assert steps > 0, "a wave does not end"
            i = rng.randrange(len(live))
            try:
                for _ in range(rng.choice((1, 1, 1, 7))):
                    next(live[i])
            except StopIteration:
                live[i] = live[-1]
                live.pop()
        return all(self.done[s] == ntasks(self.N, self.b, s) for s in range(self.N - 1))


SIZES = [(4, 16, 3, 4, 1), (17, 16, 3, 4, 2), (40, 16, 3, 4, 3), (75, 16, 3, 4, 4), (70, 32, 2, 2, 3), (120, 16, 3, 4, 5)]


@pytest.mark.parametrize("N,b,SW,R,nwg", SIZES)
def test_every_task_finds_its_blocks_and_every_wave_ends(N, b, SW, R, nwg):
    for seed in range(6):
        m = Model(N, b, SW, R, nwg)
        assert m.run(random.Random(seed)) and not m.err


@pytest.mark.parametrize("N,b,SW,R,nwg", SIZES)
@pytest.mark.parametrize("limit", [0, 3, 40])
def test_waits_that_give_up_are_flagged_and_every_wave_ends(N, b, SW, R, nwg, limit):
    for seed in range(6):
        m = Model(N, b, SW, R, nwg, limit=limit)
        assert m.run(random.Random(seed)) or m.err


def test_without_the_look_at_the_flag_the_loader_goes_round():
    with pytest.raises(AssertionError):
        for seed in range(40):
            Model(4, 16, 3, 4, 1, limit=0, check_bad=False).run(random.Random(seed), steps=20_000)


@pytest.mark.parametrize("wrong", [dict(ahead=1), dict(room=1)])
def test_looser_waits_are_seen(wrong):
    with pytest.raises(AssertionError):
        for seed in range(20):
            Model(120, 16, 3, 4, 5, **wrong).run(random.Random(seed))
