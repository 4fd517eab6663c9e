"""CPU model of the range counters of the sparse decode step (decode_kernel,
burn_dragon_amd/csrc/decode.hip): the G workgroups of a stream each add one to
the counter of its G, and the one that finds its low bits at G - 1 sums the
stream's readout.  Steps one after another must each have exactly one last
range, and steps that overlapped before them (replays of two graphs that share
a buffer, which is against the rule) must not change that.  A planted mistake
(one counter for every G, set back to zero by the range that finds G - 1) must
be caught."""
import random

import pytest


class Counters:
    def __init__(self, planted):
        self.planted = planted
        self.n = {}

    def add(self, G):
        key = 0 if self.planted else G
        old = self.n.get(key, 0)
        self.n[key] = (old + 1) % (1 << 32)
        return old

    def last(self, G, old):
        return old == G - 1 if self.planted else old % G == G - 1

    def reset(self):
        self.n[0] = 0


def _overlap(c, rnd, steps):
    """Steps of the given range counts, the ranges' operations interleaved."""
    left = []
    for G in steps:
        left += [[("add", G)] for _ in range(G)]
    while left:
        w = rnd.choice(left)
        op, *arg = w.pop()
        if op == "add":
            G = arg[0]
            old = c.add(G)
            if c.planted and c.last(G, old):
                w.append(("reset",))
        else:
            c.reset()
        if not w:
            left.remove(w)


def _step(c, G):
    return sum(c.last(G, c.add(G)) and (c.reset() if c.planted else None) is None for _ in range(G))


def _every_later_step_ends(planted, seed):
    rnd = random.Random(seed)
    c = Counters(planted)
    if not planted:
        c.n = {G: (1 << 32) - G for G in (2, 4, 8, 16, 32)}  # about to wrap
    for _ in range(4):
        for G in (32, 16, 32, 8, 4, 2):
            if _step(c, G) != 1:
                return False
        _overlap(c, rnd, rnd.choices((2, 4, 8, 16, 32), k=2))
    return all(_step(c, G) == 1 for G in (32, 16, 8, 4, 2))


@pytest.mark.parametrize("seed", range(50))
def test_overlapped_steps_spoil_no_later_step(seed):
    assert _every_later_step_ends(False, seed)


def test_planted_shared_counter_is_caught():
    assert not all(_every_later_step_ends(True, seed) for seed in range(50))
