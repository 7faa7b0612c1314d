"""Layers whose launches depend on the step: latent attention of whole contexts and of others, and a dense feed-forward in the
launches of the mixer beside it."""
import pytest
import torch

import plain_bibevik as pb
from test_gpu_parts import DEV, err, make_ctx, tensors_for

pytestmark = pytest.mark.gpu
WIDTH = 64


def latent(rt, heads=3, seed=5):
    from inferx_amd.config import PartSpec
    from inferx_amd.parts import build_part
    m = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 160, "scale": 192 ** -0.5, "rot": {"dims": 48, "base": 10000.0}}
    part = build_part("mixer", PartSpec("latent_attention", {
        "hidden_size": WIDTH, "num_heads": heads, "head_dim": 128, "rot_dim": 64, "value_dim": 128, "kv_rank": 160, "scale": m["scale"],
        "position": PartSpec("rope", {"theta": 10000.0, "rotary_dim": 48}), "init_std": 0.2}))
    w = tensors_for(part, rt, seed=seed)
    part.bind({n: t.to(DEV) for n, t in w.items()}, rt)
    plain = {n.replace(".weight", "").replace("dkv_norm", "dkv.norm"): t.double() for n, t in w.items()}
    return part, lambda x: pb.latent_attention(x.double(), plain, m, 1e-6, torch.arange(x.shape[0]))


@pytest.mark.parametrize("steps,whole", [
    ([[70, 200, 5]], [True]), ([[64]], [True]), ([[63]], [False]), ([[40, 24]], [True]), ([[1, 130, 2]], [True]),
    ([[70, 200, 5], [20, 3, 90], [1, 1, 1]], [True, False, False]),        # later steps read what the first one left in the cache
    ([[70, 200, 0], [1, 0, 150], [30, 40, 50]], [True, False, False])])    # a whole context beside one that is partly there
def test_latent_attention_layer(steps, whole, monkeypatch):
    """The layer, with its rotation and maps, against float64: keys and values of each head's own exactly where every request brings
    its whole context.  bfloat16 activations: 2e-2 of the largest, as for the other parts."""
    from inferx_amd import ops
    from inferx_amd.engine.runtime import CacheBinding, Runtime
    rt = Runtime("bfloat16")
    part, plain = latent(rt)
    calls, real = [], ops.latent_whole
    monkeypatch.setattr(ops, "latent_whole", lambda *a: calls.append(1) or real(*a))
    total = [sum(s) for s in zip(*steps)]
    x = [torch.randn(n, WIDTH, generator=torch.Generator().manual_seed(n)).to(torch.bfloat16) for n in total]
    pages = 64
    cache = CacheBinding(group=0, arrays={"latent": torch.full((pages, 1, 16, 160 + 64), float("nan"), dtype=torch.bfloat16, device=DEV)})
    outs, seen, table = [[] for _ in total], [0] * len(total), {}
    for rows, expected in zip(steps, whole):
        live = [i for i, n in enumerate(rows) if n]
        ctx, batch = make_ctx(rt, [rows[i] for i in live], [seen[i] + rows[i] for i in live], 16, pages)
        # (every request keeps pages of its own from step to step: twenty each)
        rows_of = ctx.block_tables[0].shape[1]
        ctx.block_tables[0] = torch.tensor([[20 * i + min(j, 19) for j in range(rows_of)] for i in live], dtype=torch.int32, device=DEV)
        ctx.slots[0] = torch.tensor([320 * i + p for i in live for p in range(seen[i], seen[i] + rows[i])], dtype=torch.int32, device=DEV)
        before = len(calls)
        got = part.forward(ctx, torch.cat([x[i][seen[i]:seen[i] + rows[i]] for i in live]).to(DEV), cache)
        assert len(calls) - before == (1 if expected else 0)
        for i, y in zip(live, got.cpu().split([rows[i] for i in live])):
            outs[i].append(y)
            seen[i] += rows[i]
    for i, n in enumerate(total):
        assert err(torch.cat(outs[i]), plain(x[i])) < 2e-2, f"request {i} of {n} rows"


def mixers(rt):
    from inferx_amd.config import PartSpec
    from inferx_amd.parts import build_part
    sizes = {"hidden_size": WIDTH, "num_heads": 2, "head_dim": 32, "init_std": 0.2}
    yield "latent", latent(rt)[0]
    for name, more in (("generalized_delta", {"decay_rank": 16}), ("lightning_attention", {"value_dim": 32, "decay": [0.9, 0.8]}),
                       ("retention", {"value_dim": 32, "decay": [0.9, 0.8]})):
        part = build_part("mixer", PartSpec(name, {**sizes, **more}))
        part.bind({n: t.to(DEV) for n, t in tensors_for(part, rt, seed=7).items()}, rt)
        yield name, part


@pytest.mark.parametrize("rows", [1, 8, 9, 16, 17])
@pytest.mark.parametrize("width,bias,limit", [(104, True, 7.0), (96, False, 0.0), (100, True, 0.0)])
def test_feed_forward_in_the_launches_of_the_mixer_beside_it(rows, width, bias, limit, monkeypatch):
    """Both branches of a parallel layer as they are by themselves, up to the order of 32-bit sums (a unit or two of bfloat16), for every
    mixer that takes a companion; in its launches up to sixteen rows, where the widths allow it."""
    from inferx_amd import ops
    from inferx_amd.config import PartSpec
    from inferx_amd.engine.runtime import CacheBinding, Runtime
    from inferx_amd.parts import build_part
    from inferx_amd.parts.block import ParallelBlock
    rt = Runtime("bfloat16")
    ff = build_part("feed_forward", PartSpec("dense_mlp", {"hidden_size": WIDTH, "width": width, "bias": bias, "limit": limit, "init_std": 0.2}))
    ff.bind({n: t.to(DEV) for n, t in tensors_for(ff, rt, seed=9).items()}, rt)
    norm = build_part("norm", PartSpec("rmsnorm", {"width": WIDTH, "eps": 1e-6}))
    norm.bind({"weight": torch.ones(WIDTH, dtype=torch.bfloat16, device=DEV)}, rt)
    calls, real = [], ops.linear_skinny_pair
    monkeypatch.setattr(ops, "linear_skinny_pair", lambda *a: calls.append(1) or real(*a))
    for name, mixer in mixers(rt):
        block, results = ParallelBlock({"norm": norm, "mixer": mixer, "feed_forward": ff}), []
        for takes in (False, True):
            monkeypatch.setattr(type(mixer), "takes_beside", takes)
            ctx, _ = make_ctx(rt, [1] * rows, [1] * rows, 16, 32)
            cache = CacheBinding(group=0, arrays={"latent": torch.zeros((32, 1, 16, 224), dtype=torch.bfloat16, device=DEV)})
            if name != "latent":
                cache = CacheBinding(state=torch.zeros((rows,) + tuple(mixer.state_need().shape), device=DEV))
            h = torch.randn(rows, WIDTH, generator=torch.Generator().manual_seed(rows)).to(DEV)
            del calls[:]
            results.append(block.forward(ctx, h, None, {"mixer": cache}))
            shared = takes and rows <= 16 and width % 8 == 0
            assert len(calls) == (2 if shared else 0), name
        alone, beside = results
        assert (beside.bias is None) == (alone.bias is None) == (not bias)
        for a, b in zip(alone.tensors, beside.tensors):
            assert torch.isfinite(a).all() and err(b, a.double().cpu()) < 2.0 ** -7, name
