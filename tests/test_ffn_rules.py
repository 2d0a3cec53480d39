"""The sizes the grouped FFN's host code works out for a launch, asked from the header that it takes them from. No GPU."""
import pytest

from shrike_amd import capi
from tests.helpers import ffn_rules


@pytest.mark.parametrize("tokens,top_k,experts", [(1, 1, 1), (37, 8, 256), (63, 1, 2), (64, 1, 2), (512, 8, 256), (2048, 4, 32)])
def test_no_record_is_read_past_the_tables_room(tokens, top_k, experts):
    """A bound that serves longer chunks is no promise that this chunk's table is as long."""
    pairs = tokens * top_k
    room = capi.load().shrike_hip_group_max_row_tiles(pairs, experts)
    for bound in (1, room - 1, room, room + 1, room + 1000, 0xffffffff):
        if bound:
            assert ffn_rules().readable_records(bound, pairs, experts) == min(bound, room)
