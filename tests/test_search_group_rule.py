"""How many chunks of the beam search share a compute unit (beam.hip, search_group).  A chunk that has a unit to itself takes
all its LDS: no workgroup of another decode finds room there until the search ends.  So the units that such a search leaves have to
hold a second decode of the same size.  Workgroups are dealt round eight XCDs of 32 compute units."""
import pytest

from openfish_amd import api

ALONE = 4
XCDS, UNITS = 8, 32


def per_xcd(groups):
    return -(-groups // XCDS)


def per_group(N, state_len, flags):
    return int(api.lib().ofk_search_chunks_per_group(N, state_len, flags))


@pytest.mark.parametrize("state_len", [3, 4, 5])
def test_a_lone_search_leaves_units_for_a_second_decode_of_its_size(state_len):
    chunks = 1 if state_len == 5 else 2  # of the second decode on a unit: its search, or its merged kernel
    lone = [N for N in range(1, 1025) if per_group(N, state_len, ALONE) == 1]
    assert lone == list(range(1, len(lone) + 1)) and len(lone) >= 128
    for N in lone:
        assert per_xcd(N) + per_xcd(-(-N // chunks)) <= UNITS, N


@pytest.mark.parametrize("state_len", [3, 4, 5])
def test_three_searches_that_share_the_device_find_units(state_len):
    lone = [N for N in range(1, 1025) if per_group(N, state_len, 0) == 1]
    assert lone == list(range(1, len(lone) + 1)) and len(lone) >= 32
    assert 3 * per_xcd(lone[-1]) <= UNITS


@pytest.mark.parametrize("flags", [0, ALONE])
def test_larger_batches_go_two_and_four_to_a_unit(flags):
    for state_len in (3, 4):
        assert [per_group(N, state_len, flags) for N in (256, 257, 512, 513, 2048)] == [2, 2, 2, 4, 4]
    assert [per_group(N, 5, flags) for N in (129, 256, 512, 513, 2048)] == [2, 2, 2, 2, 2]
