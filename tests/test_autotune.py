"""The schedule autotuner's choice, on an engine whose times are given."""
from types import SimpleNamespace

import ems_amd as E


class Timed:
    """What Engine.autotune reads of an engine: (H, E, whole step) ms by mode,
    and by XCD grouping."""

    def __init__(self, times, groups=None):
        self.times, self.groups, self.mode, self.group = times, groups or {}, None, None
        self.grid = SimpleNamespace(nodes=lambda: (101, 101, 101))

    def set_schedule(self, mode, tile_rows, x_chunks):
        self.mode = mode

    def set_xcd_group(self, group):
        self.group = group

    def time_kernels(self, steps):
        return self.groups.get(self.group, self.times[self.mode])


def test_ranked_by_the_whole_step():
    """The unfused step whose kernels are short and whose slab launches are
    not loses to the fused one, and wins where the whole step is shorter."""
    slow = Timed({0: (0.01, 0.01, 0.10), 1: (0.04, 0.0, 0.05), 2: (0.05, 0.0, 0.06)})
    best, trials = E.Engine.autotune(slow, xcd_groups=())
    assert best == (1, 3, 0, 0.05) and slow.mode == 1
    assert {m: ms for m, _, _, ms in trials} == {0: 0.10, 1: 0.05, 2: 0.06}
    fast = Timed({0: (0.02, 0.02, 0.045), 1: (0.03, 0.0, 0.05), 2: (0.03, 0.0, 0.06)})
    best, _ = E.Engine.autotune(fast)
    assert best == (0, 0, 0, 0.045) and fast.mode == 0 and fast.group is None


def test_groups_by_the_same_measure():
    t = Timed({0: (1.0, 1.0, 3.0), 1: (1.0, 0.0, 1.5), 2: (2.0, 0.0, 2.5)},
              {1: (0.8, 0.0, 1.6), 2: (0.9, 0.0, 1.4)})
    best, _ = E.Engine.autotune(t, xcd_groups=(1, 2))
    assert best == (1, 3, 0, 1.4) and t.group == 2
