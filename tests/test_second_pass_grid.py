"""The second pass's grid: a queue too short for the lane-per-ray kernel is
worked a wave per ray, whatever the size of the call that queued it."""
import inspect

import pytest

from psychopath_cpp_amd import gpu
from tests.cpu_build import hostbuild


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 625, 1023, 1024, 1025, 2304, 8191, 8192, 1 << 20, 2**31 - 1])
def test_a_wave_for_each_ray_of_a_short_queue(n):
    wide_min = inspect.signature(gpu.Context.set_second_pass).parameters["wide_min"].default
    longest = min(n, wide_min - 1)  # a call may queue all of its rays
    assert longest <= hostbuild.lib().hb_second_pass_waves(n) <= max(n, 1)
