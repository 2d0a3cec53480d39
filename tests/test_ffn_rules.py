"""The sizes that the host code works out for a launch, asked from the headers that it takes them from. No GPU."""
import pytest

from shrike_amd import capi
from tests import test_prefill_gpu as T
from tests.helpers import ffn_rules


@pytest.mark.parametrize("tokens,top_k,experts", [(1, 1, 1), (37, 8, 256), (63, 1, 2), (64, 1, 2), (512, 8, 256), (2048, 4, 32)])
def test_no_record_is_read_past_the_tables_room(tokens, top_k, experts):
    """A bound that serves longer chunks is no promise that this chunk's table is as long."""
    pairs = tokens * top_k
    room = capi.load().shrike_hip_group_max_row_tiles(pairs, experts)
    for bound in (1, room - 1, room, room + 1, room + 1000, 0xffffffff):
        if bound:
            assert ffn_rules().readable_records(bound, pairs, experts) == min(bound, room)


@pytest.mark.parametrize("pairs,experts,d,f,bits,shape", [
    *[(k * t, ne, d, f, bits, shape) for d, f, ne, k, t, bits, _, shape in T.SHAPE_CASES],
    *[(4 * t, ne, d, f, bits, shape) for d, f, ne, t, bits, shape in T.RING_CASES + T.EPILOGUE_CASES + T.RANGE_CASES],
    *[(2 * t, ne, d, f, bits, shape) for d, f, ne, t, bits, shape in T.TABLE_CASES],
    *[(sum(counts), len(counts), d, f, bits, shape) for counts, _, d, f, bits, shape in T.HOLE_CASES],
    *[(t, ne, d, f, bits, shape) for d, f, ne, bits, chunks in T.CHUNK_CASES for t, shape in chunks.items()]])
def test_the_gpu_tests_reach_the_shapes_they_name(pairs, experts, d, f, bits, shape):
    assert ffn_rules().routed_shape(pairs, experts, d, f, bits).decode() == shape


@pytest.mark.parametrize("experts,d,f,lines", [(128, 1024, 512, False), (128, 1024, 1024, True), (48, 2048, 1024, True), (32, 2048, 1024, False)])
def test_what_counts_against_the_cache_is_the_experts_bytes(experts, d, f, lines):
    """Cells as far apart as a caller likes are no more bytes to read: the rule is asked with what the rows' addresses are made of, and
    no spacing of whole lines changes its answer."""
    for stride in (1 << 14, 1 << 21, 1 << 25):
        assert ffn_rules().takes_lines(16 * experts, experts, d, f, 8, stride | d | f) == lines


@pytest.mark.parametrize("router_bits,widths,workgroups", [(0, (64, 2048, 4096), 4), (8, (64, 2048, 3072), 4), (4, (64, 512, 1024, 1536), 4),
                                                            (4, (1600, 2048), 3), (4, (4096,), 2)])
def test_workgroups_of_the_router_that_fit_a_compute_unit(router_bits, widths, workgroups):
    """160 KB a unit; the kernels' registers allow four."""
    for d in widths:
        assert 160 * 1024 // ffn_rules().logits_lds(router_bits, d) >= workgroups


@pytest.mark.parametrize("bits,widths,steps", [(8, (64, 512, 1024, 1088, 1280, 1536, 2112, 2304, 2560), 2), (8, (1600, 1792, 1984, 2048, 2624, 2944, 3072, 3136, 4096), 1),
                                                (4, (64, 1536, 2048, 3136, 4096), 2), (4, (2112, 2880, 3072), 1)])
def test_phase_1_walks_two_steps_where_that_was_faster(bits, widths, steps):
    for d in widths:
        assert ffn_rules().phase1_row_steps(4096, d, bits) == steps
        assert ffn_rules().phase1_row_steps(4095, d, bits) == 1
