"""The delta rules' mixers on steps that they work in chunks: their own dispatch, plans and slices, against the plain
implementations."""
import numpy as np
import pytest
import torch

import plain_bibevik as pb
import plain_dezudra as pd
from test_gpu_parts import DEV, err, make_ctx, tensors_for

pytestmark = pytest.mark.gpu

WIDTH = 64
# rows of the requests in two steps: of one row, of fewer than a chunked portion has, of several chunks; the second step
# goes on from the first one's states
STEPS = [[1, 15, 16, 200, 70], [40, 130, 1, 17, 64]]


def gated(rt):
    from inferx_amd.config import PartSpec
    from inferx_amd.parts import build_part
    m = {"heads": 4, "kv_heads": 2, "dim": 32, "vdim": 48, "conv": 4}
    part = build_part("mixer", PartSpec("gated_delta", {"hidden_size": WIDTH, "num_heads": 4, "num_kv_heads": 2, "head_dim": 32,
                                                        "value_dim": 48, "conv_taps": 4, "init_std": 0.2}))
    w = tensors_for(part, rt, seed=3)
    plain = {n.replace(".weight", ""): t.double().numpy() for n, t in w.items()}
    return part, w, lambda x: torch.from_numpy(pd.delta_mixer(x.double().numpy(), m, plain, 1e-6))


def generalized(rt):
    from inferx_amd.config import PartSpec
    from inferx_amd.parts import build_part
    m = {"heads": 3, "dim": 32}
    part = build_part("mixer", PartSpec("generalized_delta", {"hidden_size": WIDTH, "num_heads": 3, "head_dim": 32,
                                                              "decay_rank": 16, "init_std": 0.2}))
    w = tensors_for(part, rt, seed=3)
    plain = {n.replace(".weight", "").replace("a.bias", "a.b"): t.double() for n, t in w.items()}
    return part, w, lambda x: pb.general_delta(x.double(), plain, m, 1e-6)


@pytest.mark.parametrize("make,op,floats", [(gated, "delta_chunks", "delta_chunks_floats"),
                                            (generalized, "general_delta_chunks", "general_delta_floats")])
@pytest.mark.parametrize("at_a_time", [None, 2])
def test_mixers_work_long_portions_in_chunks(make, op, floats, at_a_time, monkeypatch):
    """Requests of one row to several chunks in one step, whole and in slices of two chunks (a request goes on in the next
    slice), and a second step from the states that the first one left.  bfloat16 activations: 2e-2 of the largest, as for
    the other parts; the states against those of the same mixer row by row, float32 sums in another order: 1e-5."""
    from inferx_amd import ops
    from inferx_amd.engine.runtime import CacheBinding, Runtime
    from inferx_amd.parts import delta_rule, linear_state
    rt = Runtime("bfloat16")
    part, w, plain = make(rt)
    part.bind({n: t.to(DEV) for n, t in w.items()}, rt)
    total = [a + b for a, b in zip(*STEPS)]
    x = [torch.randn(n, WIDTH, generator=torch.Generator().manual_seed(n)).to(torch.bfloat16) for n in total]
    worked = []
    real = getattr(ops, op)

    def counted(*args):
        worked.append(next(a.shape[1] for a in args if a.dim() == 2 and a.shape[0] == 2 and a.dtype == torch.int32))
        return real(*args)

    monkeypatch.setattr(ops, op, counted)
    if at_a_time:
        heads, dim, vdim = (4, 32, 48) if make is gated else (3, 32, 32)
        for module in (delta_rule, linear_state):
            monkeypatch.setattr(module, "CHUNK_WORKSPACE", at_a_time * 4 * heads * getattr(ops, floats)(dim, vdim))
    results = []
    for chunked in (False, True):
        monkeypatch.setattr(linear_state, "CHUNKS_HOST_US", -1e9 if chunked else 1e9)
        state = torch.zeros((len(total),) + tuple(part.state_need().shape), device=DEV)
        cache, outs, seen = CacheBinding(state=state), [[] for _ in total], [0] * len(total)
        for rows in STEPS:
            ctx, _ = make_ctx(rt, rows, [a + n for a, n in zip(seen, rows)], 16, 64)
            step = torch.cat([x[i][a:a + n] for i, (a, n) in enumerate(zip(seen, rows))]).to(DEV)
            for i, y in enumerate(part.forward(ctx, step, cache).cpu().split(rows)):
                outs[i].append(y)
            seen = [a + n for a, n in zip(seen, rows)]
        results.append(([torch.cat(o) for o in outs], state.cpu()))
    # chunks of the two steps' portions of at least 16 rows: 1 + 4 + 2 and 1 + 3 + 1 + 1
    assert worked == ([7, 6] if not at_a_time else [2, 2, 2, 1, 2, 2, 2])
    for i, n in enumerate(total):
        assert err(results[1][0][i], plain(x[i])) < 2e-2, f"request {i} of {n} rows"
    assert err(results[1][1], results[0][1]) < 1e-5
