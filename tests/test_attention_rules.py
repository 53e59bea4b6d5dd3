"""How many waves a workgroup of 32-bit decode attention gets, held against both forms' measured times; and which rows of a step
the bfloat16 kernels treat together: host code."""

from types import SimpleNamespace

import pytest
import torch

from bitwise_amd.csrc import ops
from bitwise_amd.engine.batch import Segment, StepContext
from bitwise_amd.parts.attention import JOIN_PARTITIONS, plan_tiles

# head size, workgroups, keys (and the most of them), microseconds in four waves, in eight
MEASURED = [(16, 64, 2400, 44.1, 33.1), (16, 256, 200, 10.3, 8.7), (16, 400, 200, 11.5, 15.1), (16, 2400, 2400, 229.8, 338.6),
            (32, 400, 20, 12.1, 10.2), (64, 2400, 60, 60.4, 52.7), (128, 2400, 4, 66.1, 51.2),
            (160, 400, 60, 10.6, 14.2), (160, 64, 800, 35.4, 25.4), (192, 1200, 20, 20.9, 30.5), (224, 64, 4, 7.0, 7.5), (224, 600, 200, 43.6, 47.4),
            (256, 256, 4, 6.9, 7.8), (256, 256, 200, 19.4, 17.6), (256, 600, 20, 13.7, 19.6), (256, 2400, 800, 616.0, 656.2)]


@pytest.mark.parametrize("head_dim,workgroups,keys,four,eight", MEASURED)
def test_the_form_that_is_taken_is_the_faster_one(head_dim, workgroups, keys, four, eight):
    waves = ops.attention_f32_waves(head_dim, workgroups, keys)
    assert {4: four, 8: eight}[waves] == min(four, eight)


def test_heads_without_a_kernel_of_four_waves_get_eight():
    for head_dim in (32, 48, 64, 80, 96, 112, 128):
        assert {ops.attention_f32_waves(head_dim, n, c) for n in (1, 256, 257, 60000) for c in (1, 64, 65, 30000)} == {8}


def tiles_of(rows, window=0, chunk=0, tokens=4, group=8, join=True):
    """Plan of requests given as (position of the first row, rows): (fold tiles, decode tiles) as lists, and the context."""
    segments = [Segment([0] * n, pos, [list(range((pos + n + 15) // 16))], i) for i, (pos, n) in enumerate(rows)]
    ctx = StepContext(segments, 1, SimpleNamespace(device=torch.device("cpu"), page_size=16))
    plan = plan_tiles(ctx, tokens, group, join, window, chunk)
    return [[] if t is None else t.tolist() for t in (plan.fold_tiles, plan.decode_tiles)], ctx


PORTION = 64 * 4          # walks 4 partitions at its last row
EDGE = 64 * (4 + JOIN_PARTITIONS)


@pytest.mark.parametrize("rows,window,chunk,joined", [
    ([(0, PORTION), (EDGE - 1, 1)], 0, 0, True), ([(0, PORTION), (EDGE, 1)], 0, 0, False),
    ([(EDGE - 1, 1), (0, PORTION), (5, 1), (200, 1)], 0, 0, True), ([(200, 1), (0, PORTION), (EDGE + 7, 1)], 0, 0, False),
    ([(0, 17), (0, PORTION), (300, 1)], 0, 0, True), ([(9000, 1), (0, PORTION)], 100, 0, True), ([(9000, 1), (0, PORTION)], 64 * 13, 0, False),
    ([(9000, 1), (0, PORTION)], 0, 256, True), ([(300, 1), (10, 1)], 0, 0, False), ([(300, 1)], 0, 0, False), ([(0, PORTION)], 0, 0, True)])
def test_single_tokens_join_a_portion_whose_walk_is_about_as_long(rows, window, chunk, joined):
    (fold, decode), ctx = tiles_of(rows, window, chunk)
    single = {ctx.seq_start[i] for i, s in enumerate(ctx.segments) if len(s.tokens) == 1 and s.pos0 + 1 >= 128}
    assert {t[0] for t in decode} == (set() if joined else single)
    # every row of the step is in one tile, a group of tiles is one request's, and the singles stand in front, the shortest first
    rows_seen = sorted(r for t in fold + decode for r in range(t[0], t[0] + t[1]))
    assert rows_seen == list(range(ctx.rows)) and len(fold) % 8 == 0
    for g in range(0, len(fold), 8):
        assert len({t[2] for t in fold[g:g + 8]}) == 1
    if joined:
        lone = [ctx.segments[t[2]].pos0 for t in fold if t[1] and len(ctx.segments[t[2]].tokens) == 1]
        assert lone == sorted(lone) and all(len(ctx.segments[t[2]].tokens) == 1 for t in fold[:8 * len(lone)])


@pytest.mark.parametrize("rows,join,same", [([(0, 300), (500, 1)], False, True), ([(0, 300), (5, 40)], True, True), ([(300, 1), (9, 1)], True, True),
                                            ([(0, 300), (9, 1), (200, 1)], True, True), ([(9000, 1), (0, 64)], True, False)])
def test_layers_whose_windows_change_nothing_share_a_plan(rows, join, same):
    """A plan is a list made on the host and a copy to the device: layers of different windows and chunks make another one only
    where it differs (here the last: with a window the far token joins the portion, without it does not)."""
    segments = [Segment([0] * n, pos, [list(range((pos + n + 15) // 16))], i) for i, (pos, n) in enumerate(rows)]
    ctx = StepContext(segments, 1, SimpleNamespace(device=torch.device("cpu"), page_size=16))
    plans = [plan_tiles(ctx, 4, 8, join, window, chunk) for window, chunk in ((0, 0), (70, 0), (128, 0), (0, 64))]
    assert all(p is plans[1] for p in plans[2:]) and (plans[0] is plans[1]) == same


# head size, key heads, (position, rows) of the longest portion, single tokens' positions (the mean of those measured), microseconds in two launches, in one
MIXES = [(128, 32, (180, 5), [360] * 230, 241.8, 289.9), (128, 32, (0, 5), [286] * 141, 128.6, 151.2), (128, 8, (0, 40), [499] * 202, 89.8, 94.8),
         (64, 32, (180, 20), [617] * 254, 231.4, 253.0), (64, 32, (490, 10), [526] * 216, 180.2, 192.4), (128, 32, (880, 6), [698] * 176, 357.9, 383.4),
         (128, 8, (0, 10), [303] * 136, 46.1, 44.1), (128, 8, (0, 190), [342] * 108, 47.2, 39.3), (64, 32, (2340, 9), [1501] * 160, 371.6, 360.4),
         (128, 8, (300, 1540), [2080] * 100, 226.1, 194.6), (64, 32, (0, 560), [544] * 76, 84.5, 78.0), (128, 8, (7850, 9), [430] * 14, 185.2, 168.4)]


@pytest.mark.parametrize("head_dim,items,portion,singles,two,one", MIXES)
def test_single_tokens_join_a_portion_where_that_is_faster(head_dim, items, portion, singles, two, one):
    segments = [Segment([0] * n, pos, [list(range((pos + n + 15) // 16))], i) for i, (pos, n) in enumerate([portion] + [(p, 1) for p in singles])]
    ctx = StepContext(segments, 1, SimpleNamespace(device=torch.device("cpu"), page_size=16))
    plan = plan_tiles(ctx, 4, 8, True, items=items, head_dim=head_dim)
    assert (plan.decode_count == 0) == (one < two) and plan.decode_count in (0, len(singles))
