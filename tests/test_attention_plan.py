"""Which kernel a step's plan gives its prompt portions to, and what the plan makes for it, on the CPU."""
import random
import types

import numpy as np
import pytest
import torch

from inferx_amd import ops
from inferx_amd.parts import attention


def step(new, seen):
    q_start = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
    return types.SimpleNamespace(memo={}, host=types.SimpleNamespace(q_start=q_start, seq_lens=np.array(seen, dtype=np.int32)),
                                 rt=types.SimpleNamespace(device="cpu"), positions=torch.arange(sum(new)))


@pytest.fixture
def card(monkeypatch):
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda device: types.SimpleNamespace(multi_processor_count=256))
    monkeypatch.setattr(ops, "upload", lambda array, device: torch.from_numpy(np.ascontiguousarray(array)))


def pays(rounds, heads, cus, slices, load):
    """What `keys_pay` says of its two times, workgroup by workgroup."""
    us = [5.5 + 1.35 * -(-r // 2) for r in rounds for _ in range(heads)]
    if not 0 < len(us) <= 2 * cus:
        return False
    ends = us[:cus]
    for i, t in enumerate(us[cus:]):  # the longest that is left follows the shortest that has run, a little later
        ends[cus - 1 - i] += 4.5 + t
    theirs = 9.3 + 1.15 * (1 + 0.1 * load) * rounds[0] if slices == 1 else 21.0 + 1.17 * rounds[0] / slices
    return 1.05 * max(ends) < theirs


def test_keys_pay_is_the_longest_place_of_all_workgroups():
    rng = random.Random(1)
    said = {True: 0, False: 0}
    for _ in range(4000):
        heads, cus = rng.choice([1, 2, 3, 16, 28, 64, 300]), rng.choice([7, 64, 256])
        tiles = rng.choice([cus // heads, cus // heads + 1, 2 * cus // heads, 2 * cus // heads + 1, rng.randint(0, 40)])  # its edges
        rounds = sorted((rng.randint(1, rng.choice([4, 40, 140])) for _ in range(tiles)), reverse=True)
        slices, load = rng.choice([1, 1, 2, 8]), rng.choice([0.0, 0.5, 1.0])
        got = attention.keys_pay(rounds, heads, cus, slices, load)
        said[got] += 1
        assert got == pays(rounds, heads, cus, slices, load), (rounds, heads, cus, slices, load)
    assert min(said.values()) > 500


def test_the_tiles_of_shared_out_keys():
    """Those of the requests' rows, the ones that read most first (in the step's order where they read as much), wherever they pay."""
    rng = random.Random(2)
    taken = 0
    for _ in range(2000):
        k, heads, slices = rng.randint(1, 5), rng.choice([1, 8, 16, 28, 64]), rng.choice([1, 1, 2, 8])
        new = [rng.randint(16, rng.choice([64, 200, 1000, 3000])) for _ in range(k)]
        seen = [n + rng.choice([0, rng.randint(0, 200), rng.randint(0, 9000)]) for n in new]
        first, seqs = [5 + sum(new[:i]) for i in range(k)], sorted(rng.sample(range(20), k))
        want = [(-(-(L - n + min(at + 64, n)) // 64), s, row + at, min(64, n - at))
                for n, L, row, s in zip(new, seen, first, seqs) for at in range(0, n, 64)]
        want.sort(key=lambda t: -t[0])
        got = attention._keys_tiles(new, seen, first, seqs, heads, 256, slices, 0.75)
        assert (got is not None) == pays([t[0] for t in want], heads, 256, slices, 0.75)
        if got is not None:
            taken += 1
            assert got.dtype == np.int32 and got.flags.c_contiguous and got.T.tolist() == [list(t[1:]) for t in want]
    assert taken > 300


@pytest.mark.parametrize("new,seen,heads,kv,keys", [([2048], [2048], 16, 16, True), ([5, 30, 60, 100, 150], [5, 30, 60, 100, 150], 16, 16, True),
                                                    ([512], [8512], 28, 4, False), ([333, 333], [1357, 1357], 28, 4, False),
                                                    ([4096], [4096], 16, 16, False)])
def test_only_the_plan_that_is_taken_is_made(card, monkeypatch, new, seen, heads, kv, keys):
    """A step's first layer waits for its plan: no tiles and pairs of the kernel that is not taken."""
    made, tiles_of, pairs = [], attention._tiles_of, attention._pairs_by_work
    monkeypatch.setattr(attention, "_tiles_of", lambda n, first, seqs, tile: made.append(tile) or tiles_of(n, first, seqs, tile))
    monkeypatch.setattr(attention, "_pairs_by_work", lambda *a, **k: made.append("pairs") or pairs(*a, **k))
    lds, waves = attention.mixed_step_plan(step(new, seen), 0, heads, kv, True, attention.WIDE_PREFILL_TILE, True)
    portions = [m for m in made if m in (64, 128, "pairs")]
    assert (lds[1] is None) == keys and portions == ([] if keys else [128, "pairs"])
    assert len(waves) == (1 if min(new) < 16 else 0)


@pytest.mark.parametrize("new,seen,heads,kv,keys", [
    ([130], [130], 16, 16, True), ([2048], [2048], 16, 16, True), ([1024], [1024], 28, 4, True), ([333], [2333], 32, 8, True),
    ([4096], [4096], 8, 8, True), ([100] * 8, [100] * 8, 16, 16, True), ([512, 512], [2512, 612], 32, 32, True),
    ([256] * 4, [256] * 4, 28, 4, False), ([100] * 8, [100] * 8, 28, 4, False), ([256] * 4, [256] * 4, 32, 32, False),
    ([384], [384], 64, 8, False), ([60, 100, 150, 30], [60, 100, 150, 30], 40, 8, False), ([1024], [1024], 40, 8, False),
    ([192], [2192], 16, 16, False), ([128], [4128], 8, 1, False), ([333, 333], [1357, 1357], 32, 8, False)])
def test_steps_at_which_both_kernels_were_timed(card, new, seen, heads, kv, keys):
    """The quicker one is taken; short prompts whose tiles of 64 queries do not all find a compute unit are left to tiles of 128."""
    lds, _ = attention.mixed_step_plan(step(new, seen), 0, heads, kv, True, attention.WIDE_PREFILL_TILE, True)
    assert (lds[1] is None) == keys
