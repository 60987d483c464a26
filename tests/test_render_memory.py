"""How many chunks a render takes in flight when device memory is short: the
rules psy_render and psy_adjoint allocate by, on the CPU."""
import pytest

from tests.cpu_build import hostbuild

OUT_OF_MEMORY, LAUNCH_FAILURE = 2, 719  # hipError_t


@pytest.mark.parametrize("want,held,room,slots,attempts", [
    (4, [], 400, 4, 1),
    (4, [], 399, 2, 2),              # two chunks when four do not fit
    (4, [], 200, 2, 2),
    (4, [100, 100, 100], 400, 4, 1),  # an earlier render's buffers are used again
    (2, [0, 100, 100], 200, 2, 2),   # those of chunks that this one has not make room for it
    (2, [100, 100, 100], 300, 2, 2),
    (1, [50, 50], 150, 1, 2),
    (4, [50, 50, 50], 200, 2, 2),
])
def test_chunks_in_flight_when_memory_is_short(want, held, room, slots, attempts):
    assert hostbuild.take_slots(want, 100, held, room) == (0, slots, attempts)


@pytest.mark.parametrize("want", [1, 2, 4])
def test_no_memory_for_two_chunks_is_an_error(want):
    rc, _, attempts = hostbuild.take_slots(want, 100, [10, 10, 10], 99)
    assert rc == OUT_OF_MEMORY and attempts <= 3


def test_other_errors_are_not_taken_for_a_shortage():
    assert hostbuild.take_slots(4, 100, [], 1000, LAUNCH_FAILURE) == (LAUNCH_FAILURE, 4, 1)


G = 1 << 30


@pytest.mark.parametrize("want,lacks,free,slots", [
    (4, [2 * G] * 4, 280 * G, 4),
    (4, [2 * G] * 4, 26 * G, 4),
    (4, [2 * G] * 4, 25 * G, 3),     # a sixteenth of the device (18 GiB) stays free
    (4, [2 * G] * 4, 21 * G, 2),
    (4, [2 * G] * 4, 1 * G, 2),      # two chunks as ever: whether they fit, the allocation says
    (4, [0, 0, 0, 0], 1 * G, 4),     # nothing to allocate
    (4, [0, 0, 0, 2 * G], 19 * G, 3),
    (2, [2 * G] * 2, 1 * G, 2),
    (1, [2 * G], 0, 1),
])
def test_more_than_two_chunks_take_plentiful_memory_only(want, lacks, free, slots):
    assert hostbuild.slots_that_fit(want, lacks, free, 288 * G) == slots
