"""The traversal autotuner's candidates, without a GPU."""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "reina-vk_amd"))
from reina_rt import autotune  # noqa: E402


class _Event:
    clock = 0.0

    def __init__(self, enable_timing=False):
        self.at = 0.0

    def record(self, stream):
        self.at = _Event.clock

    def elapsed_time(self, other):
        return other.at - self.at


class _Torch:
    class cuda:
        Event = _Event

        @staticmethod
        def synchronize():
            pass


class _Scene:
    """Queries whose time depends on the settings that reach the kernel, plus
    a little noise that would pick a winner among settings that do not."""

    def __init__(self):
        self.t = dict(stack_depth=16, refill_min=32, grid_blocks=1000, shade_blocks=4096, waves_per_simd=0)
        self.calls = 0

    def get_tuning(self):
        return dict(self.t)

    def set_tuning(self, **kw):
        self.t.update(kw)

    def intersect(self, rays, hits, n, stream=None):
        self.calls += 1
        ms = 10.0 + self.t["stack_depth"] / 16.0 + 1e-3 * (self.calls * 7919 % 13)
        if n > 1 << 18:
            ms += abs(self.t["refill_min"] - 16) + abs(self.t["grid_blocks"] - 2048) / 1024.0
        _Event.clock += ms


@pytest.mark.parametrize("n,candidates,refill,grid", [(1, 2, 32, 1000), (1 << 18, 2, 32, 1000),
                                                      ((1 << 18) + 1, 80, 16, 2048)])
def test_traversal_settings_that_do_not_reach_a_batch_stay(n, candidates, refill, grid):
    dev = _Scene()
    win, table = autotune.tune_traversal(dev, _Torch, 0, 0, n, stream=type("S", (), {"cuda_stream": 0}), cus=256)
    assert len(table) == candidates and win in table
    assert dev.t["stack_depth"] == 16 and dev.t["refill_min"] == refill and dev.t["grid_blocks"] == grid
    assert n > 1 << 18 or dev.t["waves_per_simd"] == 0
