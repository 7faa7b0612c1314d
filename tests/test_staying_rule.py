"""When the wide expert products go to workgroups that stay, on the CPU."""
import types

import pytest
import torch

from inferx_amd import ops
from inferx_amd.parts.moe import MoeFeedForward


def stays(monkeypatch, experts, top, pieces, width, hidden, tokens, gated=True):
    """Whether the grouping makes queues for this step's products."""
    part, made = MoeFeedForward(hidden, experts, top, width, pieces * width, gated=gated), []
    monkeypatch.setattr(ops, "moe_dispatch", lambda *a: made.append(a[-1]))
    rt = types.SimpleNamespace(empty=lambda shape, dtype: torch.empty(shape, dtype=dtype, device="meta"))
    part.dispatch(types.SimpleNamespace(rt=rt), torch.empty(tokens, top + pieces, dtype=torch.int32, device="meta"), ops.MOE_TILED_ROWS_WIDE, pieces)
    return made[0] is not None


@pytest.mark.parametrize("experts,top,pieces,width,hidden,tokens,expected", [
    # sizes at which whole steps were timed both ways
    (60, 4, 4, 1408, 2048, 72, False), (60, 4, 4, 1408, 2048, 100, True), (60, 4, 4, 1408, 2048, 768, True),
    (64, 8, 8, 2560, 3584, 72, False), (64, 8, 8, 2560, 3584, 96, True), (64, 8, 8, 2560, 3584, 512, True),
    (256, 8, 1, 2048, 4096, 100, False), (256, 8, 1, 2048, 4096, 768, False), (256, 8, 1, 2048, 4096, 2048, True),
    (160, 6, 2, 1536, 5120, 100, False), (160, 6, 2, 1536, 5120, 256, False), (160, 6, 2, 1536, 5120, 512, True),
    (256, 8, 1, 768, 2048, 100, True), (128, 8, 1, 1536, 4096, 100, True), (16, 2, 1, 6400, 4096, 100, True),
    # the first and the last number of tokens on either side
    (60, 4, 4, 1408, 2048, 95, False), (60, 4, 4, 1408, 2048, 96, True),
    (256, 8, 1, 2048, 4096, 1102, False), (256, 8, 1, 2048, 4096, 1103, True)])
def test_steps_whose_workgroups_stay(monkeypatch, experts, top, pieces, width, hidden, tokens, expected):
    assert stays(monkeypatch, experts, top, pieces, width, hidden, tokens) == expected


def test_products_without_a_gate_have_half_the_weights(monkeypatch):
    assert stays(monkeypatch, 256, 8, 0, 1024, 4096, 200, gated=False) and not stays(monkeypatch, 256, 8, 0, 1024, 4096, 200)


@pytest.mark.parametrize("more,fits", [({}, True), ({"hidden": 2080}, False), ({"hidden": 192}, False), ({"width": 192}, False),
                                       ({"width": 1416}, False), ({"rows2": 100, "width2": 5632}, True), ({"rows2": 100, "width2": 5640}, False),
                                       ({"rows2": 0, "width2": 5640}, True), ({"assignments": 192 * 768 - 60 * 192}, True),
                                       ({"assignments": 192 * 768}, False)])
def test_shapes_that_staying_workgroups_take(more, fits):
    assert ops.moe_stays(**{"assignments": 4096, "experts": 60, "hidden": 2048, "width": 1408, **more}) == fits


def test_the_list_of_a_dies_pairs_is_long_enough():
    """As many tiles of as many column blocks as the list holds, and one column block more."""
    experts, assignments = 8, 8
    tiles = ops.moe_max_tiles(assignments, experts, ops.MOE_TILED_ROWS_WIDE)
    blocks = 8 * (ops.MOE_QUEUE_PAIRS - ops.MOE_QUEUE_MORE) // tiles
    while tiles * (blocks + 1) // 8 + ops.MOE_QUEUE_MORE <= ops.MOE_QUEUE_PAIRS:
        blocks += 1
    for more, fits in ((0, True), (1, False)):
        assert ops.moe_stays(assignments, experts, 256, 128 * (blocks + more)) == fits
        assert ops.moe_stays(assignments, experts, 256 * (blocks + more), 256) == fits
