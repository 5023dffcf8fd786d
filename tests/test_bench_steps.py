"""bench.py times its steps as a program runs them and takes class times in builds of their own."""
import os
import sys

import numpy as np

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


class _Engine:
    def __init__(self):
        self.profiling, self.calls = True, []

    def set_profiling(self, on=True):
        self.profiling = bool(on)

    def step(self):
        self.calls.append(self.profiling)

    def class_times(self):
        assert self.profiling
        return np.array([1.0, 2.0])


def test_steps_are_timed_without_profiling():
    import bench
    e, syncs = _Engine(), []
    bench.time_steps(e, e.step, 7, 2, lambda: syncs.append(len(e.calls)))
    assert e.calls == [False] * 9
    assert syncs == [2, 9]  # both sides of the timed steps


def test_class_times_in_builds_of_their_own():
    import bench
    e = _Engine()
    assert list(bench.class_ms(e, e.step, 3)) == [1.0, 2.0]
    assert e.calls == [True] * 3 and not e.profiling
