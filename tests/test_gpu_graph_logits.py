"""Where captured steps leave their logits: written by the head's product, or copied there."""
import pytest
import torch

pytestmark = pytest.mark.gpu
VOCAB = 40008
CONFIG = {
    "architectures": ["Qwen2MoeForCausalLM"], "num_hidden_layers": 1, "hidden_size": 128, "num_attention_heads": 2,
    "num_key_value_heads": 2, "num_experts": 4, "num_experts_per_tok": 2, "moe_intermediate_size": 32,
    "shared_expert_intermediate_size": 64, "intermediate_size": 64, "decoder_sparse_step": 1, "mlp_only_layers": [],
    "norm_topk_prob": False, "vocab_size": VOCAB, "rope_theta": 10000.0, "rms_norm_eps": 1e-6,
    "max_position_embeddings": 64, "use_sliding_window": False, "tie_word_embeddings": False}


@pytest.mark.parametrize("scale", [1.0, 0.25])
@pytest.mark.parametrize("dtype,requests,in_place", [
    ("bfloat16", 2, True), ("bfloat16", 17, True), ("bfloat16", 33, True), ("bfloat16", 65, False),  # (the last: the library's)
    ("float32", 17, True), ("float32", 33, False)])
def test_captured_steps_leave_the_logits_of_uncaptured_ones(dtype, requests, in_place, scale):
    """Two shapes whose graphs share the buffer, replayed in turn with other tokens each time, against a runner without graphs: the same
    bits, and what was returned before stays as it is."""
    from inferx_amd.config import config_from_dict
    from inferx_amd.engine.batch import build_step_batch
    from inferx_amd.engine.runner import ModelRunner
    from inferx_amd.engine.runtime import Runtime
    from inferx_amd.parts import build_model
    config = config_from_dict(CONFIG)
    rt = Runtime(dtype)
    gen = torch.Generator().manual_seed(3)

    def runner():
        model = build_model(config.model_spec())
        gen.manual_seed(3)
        weights = {n: rt.place((torch.ones(p.shape) if p.init == "ones" else torch.randn(p.shape, generator=gen) * 0.1).to(rt.dtype))
                   for n, p in model.expected_tensors().items()}
        r = ModelRunner(config, weights, rt, num_pages=requests + 1, max_requests=requests, max_seq_len=16, model=model)
        r.model.head.scale = scale
        for i in range(requests):
            r.add_request(i)
        r.run_entries([(i, [7 + i, 11 * i % VOCAB], []) for i in range(requests)])
        return r

    def step(r, n, turn):
        return r.step(build_step_batch(r.cache, [(i, [(1000 * turn + 13 * i) % VOCAB], [0]) for i in range(n)]))

    eager, captured = runner(), runner()
    captured.capture_after = 1
    places, forward = [], captured.model.forward
    captured.model.forward = lambda ctx, bindings: places.append(forward(ctx, bindings)) or places[-1]
    kept = []
    for turn in range(4):
        for n in (requests, requests - 1):
            places.clear()
            got = step(captured, n, turn)
            if turn == 0:  # (a run that warms up, and the recorded one)
                mine = captured._graph_logits.data_ptr()
                if n == requests:
                    assert [p.data_ptr() == mine for p in places] == [in_place] * 2
            assert (turn == 0) == bool(places)
            places.clear()
            eager._graph_uses.clear()  # (a shape's first step runs kernel by kernel with the plans of the recorded one)
            kept.append((got, step(eager, n, turn)))
            assert not eager._graphs and torch.isfinite(got).all()
    for got, want in kept:
        assert torch.equal(got, want)
    assert not torch.equal(kept[0][0], kept[2][0])
