"""How the rows of a step's requests are cut into the chunks of the recurrences' chunked forms, on the CPU."""
from types import SimpleNamespace as NS

import numpy as np
import pytest
import torch

from inferx_amd import ops
from inferx_amd.parts import delta_rule, linear_state


@pytest.fixture
def cpu(monkeypatch):
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda t: t)


def step(lengths):
    starts = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    return NS(one_token_each=False, memo={}, host=NS(q_start=starts), rt=NS(device=torch.device("cpu")))


LENGTHS = [[1, 15, 16, 200, 70], [64], [65, 0, 63, 129, 16, 15], [17] * 9, [1000, 3, 500], [2, 1, 15]]


@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("most", [1, 2, 3, 7, 1000])
def test_chunk_slices_hold_every_row_of_long_portions_once_and_in_order(lengths, most, cpu):
    ctx, starts = step(lengths), np.concatenate([[0], np.cumsum(lengths)])
    at = {s: int(starts[s]) for s, n in enumerate(lengths) if n >= linear_state.CHUNKED_MIN_ROWS}  # the next row of each
    slices = linear_state.chunk_slices(ctx, linear_state.CHUNKED_MIN_ROWS, most)
    for chunks, seqs in slices:
        assert chunks.dtype == seqs.dtype == torch.int32 and 0 < chunks.shape[1] <= most
        row0, rows = chunks.tolist()
        seen = 0
        for s, first, count in zip(*seqs.tolist()):
            assert first == seen and count > 0, "a slice's requests have its chunks one after the other"
            for c in range(first, first + count):
                assert row0[c] == at[s] and 0 < rows[c] <= ops.LINEAR_CHUNK_ROWS
                assert rows[c] == ops.LINEAR_CHUNK_ROWS or row0[c] + rows[c] == starts[s + 1], "only a last chunk is short"
                at[s] += rows[c]
            seen += count
        assert seen == chunks.shape[1]
    assert at == {s: int(starts[s + 1]) for s in at}
    assert linear_state.shorter_portions(ctx, linear_state.CHUNKED_MIN_ROWS) == any(0 < n < 16 for n in lengths)
    chunks, seqs, others = linear_state.chunk_plan(ctx)
    assert others == any(0 < n < 16 for n in lengths) and (chunks is None) == (not at)
    if chunks is not None:
        assert chunks.shape[1] == sum(c.shape[1] for c, _ in slices)


@pytest.mark.parametrize("costs,heads,dim,vdim,lengths,chunked", [
    # measured on one card, us row by row and in chunks: what is clearly faster is taken, what is slower is not
    (delta_rule.GATED_COSTS, 16, 128, 128, [128], False),           # 46, 51
    (delta_rule.GATED_COSTS, 16, 128, 128, [448], True),            # 150, 75
    (delta_rule.GATED_COSTS, 16, 128, 128, [64] * 32, True),        # 336, 176
    (delta_rule.GATED_COSTS, 16, 64, 64, [160] * 8, False),         # 48, 60
    (delta_rule.GATED_COSTS, 4, 128, 256, [200] * 4, False),        # 72, 85
    (linear_state.CORRECTED_COSTS, 32, 64, 64, [128], False),       # 35, 39
    (linear_state.CORRECTED_COSTS, 32, 64, 64, [2048], True),       # 493, 167
    (linear_state.CORRECTED_COSTS, 32, 32, 32, [160] * 32, False),  # 69, 231
    (linear_state.CORRECTED_COSTS, 32, 32, 32, [640] * 8, False),   # 113, 193
    (linear_state.CORRECTED_COSTS, 16, 128, 128, [200], False),     # 71, 87
    (delta_rule.GATED_COSTS, 16, 48, 48, [2048], False),            # (a size that has no chunked form)
    (delta_rule.GATED_COSTS, 16, 128, 128, [15] * 200, False)])     # (no portion that is worked in chunks)
def test_which_steps_are_worked_in_chunks(costs, heads, dim, vdim, lengths, chunked):
    assert linear_state.chunks_pay(step(lengths), heads, dim, vdim, costs) == chunked
    one = NS(one_token_each=True, memo={}, host=None)
    assert not linear_state.chunks_pay(one, heads, dim, vdim, costs)
