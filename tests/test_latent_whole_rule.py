"""Which steps latent attention works on keys and values of each head's own, the tiles it makes for them, and when slices of keys are
merged in the launch of the value maps, on the CPU."""
import types

import numpy as np
import pytest
import torch

from inferx_amd import ops
from inferx_amd.csrc import build
from inferx_amd.parts.latent_attention import LatentAttention


def part_for(heads=2, w_kv=True, **more):
    part = LatentAttention(64, heads, 128, 64, 128, 512, **more)
    part.w_kv = torch.empty(0) if w_kv else None  # (only whether they are there is looked at)
    part.w_in = torch.empty(heads * 192 + 576, 0)
    return part


def step(new, seen, **more):
    q_start = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
    ctx = types.SimpleNamespace(memo={}, host=types.SimpleNamespace(q_start=q_start, seq_lens=np.array(seen, dtype=np.int32)),
                                rt=types.SimpleNamespace(device="cpu"), num_tokens=sum(new), one_token_each=False)
    ctx.__dict__.update(more)
    return ctx


@pytest.fixture(autouse=True)
def no_card(monkeypatch):
    monkeypatch.setattr(ops, "upload", lambda array, device: torch.from_numpy(np.ascontiguousarray(array)))


WRITES, READS = types.SimpleNamespace(writes=True), types.SimpleNamespace(writes=False)


def test_tiles_of_whole_contexts():
    """First row, rows and position of up to 64 queries each; those that read most keys first; nothing of a request without rows."""
    tiles = part_for().whole_contexts(step([70, 0, 200, 1], [70, 9, 200, 1]), None, WRITES)
    assert tiles.t().tolist() == [[70 + 192, 8, 192], [70 + 128, 64, 128], [70 + 64, 64, 64], [64, 6, 64], [0, 64, 0], [70, 64, 0], [270, 1, 0]]


@pytest.mark.parametrize("new,seen,whole", [([64], [64], True), ([63], [63], False), ([40, 24], [40, 24], True), ([40, 24], [40, 25], False),
                                            ([64, 100], [65, 100], False), ([64, 0], [64, 30], True)])
def test_steps_of_whole_contexts(new, seen, whole):
    assert (part_for().whole_contexts(step(new, seen), None, WRITES) is not None) == whole


@pytest.mark.parametrize("change", ["window", "head gate", "reads", "one token each", "captured", "scale", "other sizes", "rows of q"])
def test_what_keeps_a_step_on_the_latents(change):
    part = part_for(w_kv=change != "other sizes", **{"window": {"window": 100}, "head gate": {"head_gate": True}, "scale": {"scale": -1.0}}.get(change, {}))
    if change == "rows of q":
        part.w_in = torch.empty(2 * 192 + 576 + 4, 0)
    ctx = step([100], [100], **{"one token each": {"one_token_each": True}, "captured": {"host": None}}.get(change, {}))
    assert part_for().whole_contexts(step([100], [100]), None, WRITES) is not None
    assert part.whole_contexts(ctx, None, READS if change == "reads" else WRITES) is None


@pytest.mark.parametrize("heads,tokens,fits", [(32767, 64, True), (32768, 64, False), (16, (1 << 19) - 1, True), (16, 1 << 19, False)])
def test_sizes_that_places_within_keys_and_values_hold(heads, tokens, fits):
    """Rows' places are 24-bit numbers multiplied, 32 bits in all: other sizes are refused, and go the other way."""
    part = part_for(1)
    part.num_heads = heads
    assert (part.whole_contexts(step([tokens], [tokens]), None, WRITES) is not None) == fits
    refused = build.load().ix_latent_whole(None, 0, 0, None, None, None, 0, None, 0, 0, tokens, heads, 1.0, None)  # no tiles
    assert (refused == 0) == fits


@pytest.mark.parametrize("tokens,heads,n,rank,slices,together", [
    (1, 16, 128, 512, 32, True), (16, 16, 128, 512, 16, True), (16, 17, 128, 512, 16, False), (2, 128, 128, 512, 32, True),
    (16, 128, 128, 512, 8, False), (16, 32, 64, 256, 16, True), (16, 33, 64, 256, 16, False), (16, 32, 64, 264, 16, False),
    (8, 16, 128, 512, 1, False)])
def test_slices_are_merged_where_their_products_are_formed_only_for_few_pairs(monkeypatch, tokens, heads, n, rank, slices, together):
    """One workgroup a token and head reads the head's whole map."""
    part, done = LatentAttention(64, heads, 128, 64, n, rank), []
    monkeypatch.setattr(ops, "latent_mfma_fits", lambda *a: True)
    monkeypatch.setattr(ops, "latent_mfma_splits", lambda *a: slices)
    monkeypatch.setattr(ops, "latent_attention_mfma", lambda *a: done.append(a[-1]))
    monkeypatch.setattr(ops, "latent_merge_product", lambda *a: done.append("merged"))
    meta = lambda *shape, dtype=torch.bfloat16: torch.empty(shape, dtype=dtype, device="meta")
    ctx = step([1] * tokens, [100] * tokens, one_token_each=True, block_tables=[None], seq_of_token=None, positions=None)
    ctx.rt.empty = lambda shape, dtype: meta(*shape, dtype=dtype)
    cache = types.SimpleNamespace(arrays={"latent": None}, group=0)
    got = part.attend(ctx, meta(tokens, heads, rank), None, cache, meta(tokens, heads, rank), None, meta(tokens, heads, n))
    assert got == together and done == ([False, "merged"] if together else [True])
