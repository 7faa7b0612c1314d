"""What is timed when the engine's speed is judged: the steps that a serving or batch program has it do.

A case is one model at its real layer sizes (fewer layers: every layer of a kind costs the same) with random weights,
and one pass of work through `ModelRunner`, the step function that the engine, the trace replay and the benchmark call:

    decode     one token for each of `requests` requests whose contexts are there already
    mixed      the same beside `portions` prompt portions of `portion` tokens on contexts of `before`
    prompts    `requests` whole prompts in one step, from adding the requests to ending them
    generate   `requests` prompts in one step, then `new` steps of one token each, as the replay of a trace does it

Lengths of contexts and prompts are spread evenly in their logarithm from `shortest` to `longest`.  The models:

    a27b, 57b   Qwen2-MoE at the sizes of Qwen1.5-MoE-A2.7B (16 heads with keys of their own) and Qwen2-57B-A14B
                (28 heads on 4 sets of keys), the architecture that the engine is built around
    dezudra     the gated delta rule and differential attention over a window in turn, without the feed-forwards
                (its norm after the experts carries a near tie between two of them through the whole model, so that
                two correct runs differ by more than a wrong one would show)
    bibevik     the generalized delta rule, lightning attention and latent attention, clamped dense feed-forwards;
                its mixers' kernels are also those of the other designs' recurrences and latent attention

Tokens are given, not sampled, so that a pass computes the same whichever of two near-equal logits wins.
"""
from __future__ import annotations

import math
import zlib

import torch

from inferx_amd.config import config_from_dict
from inferx_amd.engine.batch import build_step_batch
from inferx_amd.engine.runner import ModelRunner
from inferx_amd.engine.runtime import Runtime
from inferx_amd.parts import build_model

F64 = torch.float64
PAGE = 16


# ---- the cases ----------------------------------------------------------------------------------------------------
def _case(name, do, model, layers, requests, shortest, longest, dtype="bfloat16", portions=0, portion=0, before=0, new=0,
          wanted=1):
    case = {"do": do, "model": model, "layers": layers, "dtype": dtype, "requests": requests, "shortest": shortest,
            "longest": longest, "portions": portions, "portion": portion, "before": before, "new": new, "wanted": wanted}
    return case if name is None else dict(case, name=name)


def listed():
    return [
        # one conversation: the latency of a token, launches and the smallest products
        _case("decode_1", "decode", "a27b", 8, 1, 517, 517),
        # the benchmark's headline: eight requests behind prompts of 2,048 tokens
        _case("decode_8", "decode", "a27b", 8, 8, 2048, 2048),
        # a full server: 64 requests that are differently far along
        _case("decode_64", "decode", "a27b", 8, 64, 200, 2048),
        # a long prompt read in one step, its last 16 positions scored
        _case("prompt_2048", "prompts", "a27b", 8, 1, 2048, 2048, wanted=16),
        # short prompts that arrive together, of ragged lengths
        _case("prompts_short", "prompts", "a27b", 8, 7, 5, 150),
        # chunked reading of a long document under a token budget, grouped heads
        _case("portion_on_8k", "mixed", "57b", 4, 0, 0, 0, portions=1, portion=512, before=8000, wanted=16),
        # a server between admissions: decoding beside two prompt portions
        _case("mixed_57b", "mixed", "57b", 4, 16, 700, 3000, portions=2, portion=333, before=1024),
        # 32-bit runs, those that results are checked against
        _case("decode_8_float32", "decode", "a27b", 4, 8, 300, 1200, dtype="float32"),
        _case("prompts_float32", "prompts", "a27b", 4, 2, 150, 361, dtype="float32", wanted=4),
        # the other designs' mixers: ragged prompts, one long prompt, and prompts with the tokens that follow
        _case("dezudra_prompts", "prompts", "dezudra", 4, 2, 611, 1437, wanted=8),
        _case("bibevik_prompt", "prompts", "bibevik", 4, 1, 2048, 2048, wanted=16),
        _case("bibevik_generate", "generate", "bibevik", 4, 8, 40, 200, new=16),
    ]


def draw(rng):
    """One more case of the ranges that the listed ones span; sizes are spread over their logarithm."""
    span = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.choice(("decode", "decode", "prompts", "prompts", "portion", "mixed", "float32", "dezudra", "bibevik", "generate"))
    if kind == "decode":
        shortest = span(16, 1024)
        return _case(None, "decode", "a27b", 8, span(1, 64), shortest, span(shortest, 2048))
    if kind == "prompts":
        n = span(1, 8)
        shortest = span(3, 400 // n)
        return _case(None, "prompts", "a27b", 8, n, shortest, span(shortest, 2048 // n), wanted=min(shortest, 4))
    if kind == "portion":
        return _case(None, "mixed", "57b", 4, 0, 0, 0, portions=1, portion=span(17, 512), before=span(300, 8000), wanted=16)
    if kind == "mixed":
        shortest = span(64, 1024)
        return _case(None, "mixed", "57b", 4, span(2, 16), shortest, span(shortest, 3000), portions=span(1, 2),
                     portion=span(17, 333), before=span(64, 1024))
    if kind == "float32":
        if rng.random() < 0.5:
            return _case(None, "decode", "a27b", 4, span(1, 8), 200, span(200, 1200), dtype="float32")
        n = span(1, 2)
        return _case(None, "prompts", "a27b", 4, n, span(9, 150), span(151, 361), dtype="float32", wanted=4)
    if kind == "generate":
        model = rng.choice(("dezudra", "bibevik"))
        return _case(None, "generate", model, 4, span(1, 8), span(20, 60), span(61, 200), new=rng.randint(8, 16))
    n = span(1, 3)
    shortest = span(20, 600 // n)
    return _case(None, "prompts", kind, 4, n, shortest, span(shortest, 2048 // n), wanted=8)


def _lengths(case):
    n, lo, hi = case["requests"], case["shortest"], case["longest"]
    return [int(round(lo * (hi / lo) ** (i / (n - 1)))) if n > 1 else hi for i in range(n)]


# ---- the models ---------------------------------------------------------------------------------------------------
def _config(case):
    """What config.json holds."""
    L = case["layers"]
    if case["model"] in ("a27b", "57b"):
        small = case["model"] == "a27b"
        return {"architectures": ["Qwen2MoeForCausalLM"], "num_hidden_layers": L, "hidden_size": 2048 if small else 3584,
                "num_attention_heads": 16 if small else 28, "num_key_value_heads": 16 if small else 4, "head_dim": 128,
                "num_experts": 60 if small else 64, "num_experts_per_tok": 4 if small else 8,
                "moe_intermediate_size": 1408 if small else 2560,
                "shared_expert_intermediate_size": 5632 if small else 20480, "intermediate_size": 5632,
                "decoder_sparse_step": 1, "mlp_only_layers": [], "norm_topk_prob": False, "vocab_size": 151936,
                "rope_theta": 1000000.0, "rms_norm_eps": 1e-6, "max_position_embeddings": 32768,
                "use_sliding_window": False, "tie_word_embeddings": False}
    W, H, D = 2048, 16, 128
    if case["model"] == "dezudra":
        delta = {"type": "delta", "mlp": None, "mixer": {"heads": H, "kv_heads": 4, "dim": D, "vdim": D, "conv": 4}}
        attention = {"type": "attention", "mlp": None,
                     "mixer": {"heads": H, "kv_heads": 4, "dim": D // 2, "vdim": D, "conv": 4, "scale": (D // 2) ** -0.5,
                               "diff": 0.5, "rot": {"dims": D // 2, "base": 10000.0}, "mask": {"size": 1024, "keep_first": 4}}}
        return {"architecture": "Dezudra", "vocab": 32000, "width": W, "norm": {"eps": 1e-6}, "logit_scale": 1.0,
                "layers": [(delta, attention)[i % 2] for i in range(L)]}
    mlp = {"kind": "dense", "ff": 5632, "limit": 7.0}
    latent = {"type": "latent_attention", "mlp": mlp,
              "mixer": {"heads": H, "dim": D, "rot_dim": 64, "vdim": D, "kv_rank": 512, "scale": (D + 64) ** -0.5,
                        "rot": {"dims": 64, "base": 10000.0}}}
    delta = {"type": "general_delta", "mlp": mlp, "mixer": {"heads": 32, "dim": 64, "decay_rank": 64}}
    lightning = {"type": "lightning", "mlp": mlp,
                 "mixer": {"heads": H, "dim": D, "vdim": D, "decay": [1.0 - 2.0 ** (-5 - 3 * h / H) for h in range(H)]}}
    return {"architecture": "Bibevik", "vocab": 32000, "width": W, "norm": {"eps": 1e-6}, "embedding": {"scale": 1.0},
            "layers": [(delta, latent, lightning, latent)[i % 4] for i in range(L)]}


def _weights(case, model, seed):
    """Checkpoint name -> tensor on the device, in the storage type; a tensor is a function of the seed and its name."""
    dtype = getattr(torch, case["dtype"])
    gen = torch.Generator(device="cuda")
    out = {}
    for name, p in model.expected_tensors().items():
        gen.manual_seed((zlib.crc32(name.encode()) << 16) + seed % 65536)
        t = torch.randn(p.shape, generator=gen, device="cuda", dtype=dtype)
        out[name] = t.mul_(0.1).add_(1.0) if p.init == "ones" else t.mul_(p.std).add_(p.mean)
    return out


def _tokens(case, seed):
    """Per request, then per portion, its tokens: the context with the step's own token, the prompt with what follows, the
    portion with what is before it."""
    gen = torch.Generator().manual_seed(seed)
    extra = {"decode": 1, "mixed": 1, "prompts": 0, "generate": case["new"]}[case["do"]]
    lengths = [n + extra for n in _lengths(case)] if case["requests"] else []
    lengths += [case["before"] + case["portion"]] * case["portions"]
    vocab = 151936 if case["model"] in ("a27b", "57b") else 32000
    return [torch.randint(0, vocab, (n,), generator=gen).tolist() for n in lengths]


def prepare(case, seed):
    config = config_from_dict(_config(case))
    rt = Runtime(case["dtype"], "cuda:0")
    model = build_model(config.model_spec())
    weights = _weights(case, model, seed)
    tokens = _tokens(case, seed)
    pages = [-(-len(t) // PAGE) + 1 for t in tokens]
    runner = ModelRunner(config, weights, rt, page_size=PAGE, num_pages=sum(pages), max_requests=len(tokens),
                         max_seq_len=max(pages) * PAGE, model=model)
    state = {"case": case, "runner": runner, "tokens": tokens}
    if case["do"] in ("decode", "mixed"):  # the contexts are read, in steps of at most 4,096 tokens
        known = [len(t) - (1 if i < case["requests"] else case["portion"]) for i, t in enumerate(tokens)]
        entries, room = [], 4096
        for i, n in enumerate(known):
            runner.add_request(i)
            at = 0
            while at < n:
                m = min(n - at, room)
                entries.append((i, tokens[i][at:at + m], []))
                at, room = at + m, room - m
                if room == 0:
                    runner.run_entries(entries)
                    entries, room = [], 4096
        if entries:
            runner.run_entries(entries)
        rows = lambda i: [0] if i < case["requests"] else list(range(case["portion"] - case["wanted"], case["portion"]))
        state["entries"] = [(i, tokens[i][n:], rows(i)) for i, n in enumerate(known)]
        if case["do"] == "decode":  # a server has met this shape before
            for _ in range(runner.capture_after):
                run(state)
    return state


def run(state):
    case, runner, tokens = state["case"], state["runner"], state["tokens"]
    if case["do"] in ("decode", "mixed"):
        # laid out and run, but not committed: the next pass takes the same step again
        return runner.step(build_step_batch(runner.cache, state["entries"]))
    for i in range(len(tokens)):
        runner.add_request(i)
    n = [len(t) - case["new"] for t in tokens]
    out = [runner.run_entries([(i, t[:n[i]], list(range(n[i] - case["wanted"], n[i]))) for i, t in enumerate(tokens)])]
    for k in range(case["new"]):
        out.append(runner.run_entries([(i, t[n[i] + k:n[i] + k + 1], [0]) for i, t in enumerate(tokens)]))
    for i in range(len(tokens)):
        runner.end_request(i)
    return out


# ---- what a pass cannot do without ----------------------------------------------------------------------------------
def work(case):
    """Every weight that the pass's tokens use, read once per step (the experts that an even router gives them), what the
    step reads of its contexts, the logits written; the products' and the attention's operations."""
    cfg, L = _config(case), case["layers"]
    elt = 2 if case["dtype"] == "bfloat16" else 4
    lengths = _lengths(case) if case["requests"] else []
    if case["do"] in ("decode", "mixed"):
        steps = [[(1, n) for n in lengths] + [(case["portion"], case["before"])] * case["portions"]]
        rows = len(lengths) + case["portions"] * case["wanted"]
    else:
        steps = [[(n, 0) for n in lengths]] + [[(1, n + k) for n in lengths] for k in range(case["new"])]
        rows = len(lengths) * case["wanted"]
    total_bytes = total_flops = 0.0
    for s, step in enumerate(steps):
        T = sum(new for new, _ in step)
        seen = lambda window: sum(min(old + new, window or old + new) if new == 1 else old + new for new, old in step)
        pairs = lambda window: sum(new * old + new * (new + 1) / 2 if not window else
                                   sum(min(old + i + 1, window) for i in range(new)) for new, old in step)
        R = rows if s == 0 else len(lengths)
        if case["model"] in ("a27b", "57b"):
            H, D = cfg["hidden_size"], 128
            qd, kvd = cfg["num_attention_heads"] * D, cfg["num_key_value_heads"] * D
            E, k, mi, si = (cfg[n] for n in ("num_experts", "num_experts_per_tok", "moe_intermediate_size",
                                             "shared_expert_intermediate_size"))
            fixed = L * ((2 * qd + 2 * kvd) * H + E * H + 3 * si * H)
            experts, per_token = L * E * (1 - (1 - k / E) ** T) * 3 * mi * H, L * k * 3 * mi * H
            cache, attention = L * 2 * kvd * seen(0), L * 4 * qd * pairs(0)
        else:
            H = cfg["width"]
            fixed = experts = per_token = cache = attention = 0.0
            for layer in cfg["layers"]:
                m = layer["mixer"]
                if layer["type"] in ("delta", "general_delta", "lightning"):
                    G, D = m.get("kv_heads", m["heads"]), m["dim"]
                    qk, v = G * D, m["heads"] * m.get("vdim", D)
                    fixed += H * (2 * qk + 3 * v + (v if layer["type"] == "general_delta" else 0))
                    attention += 6.0 * T * v * D  # the state's decay, update and read, a number of it for each
                    cache += 2 * 4 / elt * len(step) * v * D  # the state, in 32 bits, read and written
                elif layer["type"] == "attention":
                    qd, kd, v = 2 * m["heads"] * m["dim"], 2 * m["kv_heads"] * m["dim"], m["kv_heads"] * m["vdim"]
                    fixed += H * (qd + kd + v + m["heads"] * m["vdim"])
                    attention += 2.0 * pairs(m["mask"]["size"]) * (qd + 2 * m["heads"] * m["vdim"])
                    cache += (kd + v) * seen(m["mask"]["size"])
                else:
                    rank, D, heads = m["kv_rank"], m["dim"], m["heads"]
                    fixed += H * (heads * (D + 64) + rank + 64 + heads * D) + 2 * heads * D * rank
                    attention += 2.0 * pairs(0) * heads * (2 * D + 64)
                    cache += (rank + 64) * seen(0)
                fixed += 3 * H * layer["mlp"]["ff"] if layer["mlp"] else 0
        vocab = cfg.get("vocab_size") or cfg["vocab"]
        total_bytes += (fixed + experts + vocab * H + cache + T * H) * elt + 4 * R * vocab
        total_flops += 2.0 * T * (fixed + per_token) + 2.0 * R * vocab * H + attention
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case):
    """Four times what was seen: 32-bit runs are 6e-6 off the 64-bit result (most of it the angles of the rotation, which
    are 32-bit); bfloat16 runs with other sums are 0.006 to 0.011 apart with experts, where near ties in the router fall
    either way, at most 0.09 of the root mean square in one place, and the designs without experts are 0.007 off the
    64-bit result."""
    if case["dtype"] == "float32":
        return {"rel": 3e-5, "max": 1e-3}
    return {"rel": 0.03, "max": 0.4} if case["model"] in ("a27b", "57b") else {"rel": 0.02, "max": 0.2}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------------
class _Plain:
    """A pass's logits in float64 by plain torch: whole sequences, no cache."""

    def __init__(self, case, seed):
        self.cfg, self.case = _config(case), case
        self.w = _weights(case, build_model(config_from_dict(self.cfg).model_spec()), seed)

    def __getitem__(self, name):
        return self.w[name].to(F64)

    def linear(self, x, name):
        return x @ self[name].T

    @staticmethod
    def unit(x, eps):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)

    def norm(self, x, name):
        return self.unit(x, 1e-6) * self[name]

    @staticmethod
    def angles(T, dims, base):
        a = torch.arange(T, device="cuda", dtype=F64)[:, None] * base ** (-2.0 * torch.arange(dims // 2, device="cuda", dtype=F64) / dims)
        return torch.cos(a)[:, None, :], torch.sin(a)[:, None, :]

    def rotate(self, x, dims, base):
        """x [T, heads, d]: pairs (i, i + dims / 2)."""
        c, s = self.angles(x.shape[0], dims, base)
        u, v = x[..., :dims // 2], x[..., dims // 2:dims]
        return torch.cat([u * c - v * s, v * c + u * s, x[..., dims:]], -1)

    def rotate_neighbours(self, x, dims, base):
        """x [T, heads, d]: pairs (2 i, 2 i + 1)."""
        c, s = self.angles(x.shape[0], dims, base)
        u, v = x[..., 0:dims:2], x[..., 1:dims:2]
        return torch.stack([u * c - v * s, v * c + u * s], -1).reshape(x.shape)

    @staticmethod
    def attend(q, k, v, scale, window=0, keep_first=0):
        """q [T, heads, d], k [T, kv heads, d], v [T, kv heads, e] -> [T, heads, e], a block of queries at a time."""
        T, heads, _ = q.shape
        rep = heads // k.shape[1]
        k, v = (t.permute(1, 0, 2).repeat_interleave(rep, 0).contiguous() for t in (k, v))
        j, out = torch.arange(T, device="cuda"), []
        for at in range(0, T, 512):
            i = j[at:at + 512, None]
            seen = (j <= i) & ((i - j < window) | (j < keep_first)) if window else j <= i
            s = q[at:at + 512].permute(1, 0, 2).contiguous() @ k.transpose(1, 2).contiguous()
            out.append((torch.softmax((s * scale).masked_fill(~seen, -math.inf), -1) @ v).permute(1, 0, 2))
        return torch.cat(out)

    def experts(self, x, weights, ids, f):
        """sum over the slots of weight * f(expert, its rows)."""
        out = torch.zeros_like(x)
        for e in ids.unique().tolist():
            row, slot = torch.nonzero(ids == e, as_tuple=True)
            out.index_add_(0, row, weights[row, slot, None] * f(e, x[row]))
        return out

    # the layers: x of all sequences one after the other, `parts` their slices
    def qwen(self, h, parts):
        c = self.cfg
        heads, kv = c["num_attention_heads"], c["num_key_value_heads"]
        silu = torch.nn.functional.silu
        for l in range(c["num_hidden_layers"]):
            p = f"model.layers.{l}."
            x, a = self.norm(h, p + "input_layernorm.weight"), p + "self_attn."
            q, k, v = (self.linear(x, a + n + "_proj.weight") + self[a + n + "_proj.bias"] for n in "qkv")
            o = torch.cat([self.attend(self.rotate(q[s].view(-1, heads, 128), 128, c["rope_theta"]),
                                       self.rotate(k[s].view(-1, kv, 128), 128, c["rope_theta"]),
                                       v[s].view(-1, kv, 128), 128 ** -0.5) for s in parts])
            h = h + self.linear(o.reshape(len(h), -1), a + "o_proj.weight")
            x, m = self.norm(h, p + "post_attention_layernorm.weight"), p + "mlp."
            mlp = lambda x, n: self.linear(silu(self.linear(x, n + "gate_proj.weight")) * self.linear(x, n + "up_proj.weight"),
                                           n + "down_proj.weight")
            weights, ids = torch.softmax(self.linear(x, m + "gate.weight"), -1).topk(c["num_experts_per_tok"], -1)
            h = h + self.experts(x, weights, ids, lambda e, rows: mlp(rows, f"{m}experts.{e}."))
            h = h + torch.sigmoid(self.linear(x, m + "shared_expert_gate.weight")) * mlp(x, m + "shared_expert.")
        return h, "model.norm.weight", "lm_head.weight"

    @staticmethod
    def conv(x, w):
        taps = w.shape[1]
        padded = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
        return sum(padded[j:j + len(x)] * w[:, j] for j in range(taps))

    def gated_delta(self, x, p, m):
        T, H, G, D, V = len(x), m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        silu = torch.nn.functional.silu
        q, k, v = (silu(self.conv(self.linear(x, p + n), self[p + n + ".conv"])) for n in "qkv")
        q, k = q.view(T, G, D), k.view(T, G, D)
        q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6) * D ** -0.5
        k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        q, k, v = q.repeat_interleave(H // G, 1), k.repeat_interleave(H // G, 1), v.view(T, H, V)
        beta = torch.sigmoid(self.linear(x, p + "b"))
        g = torch.exp(-torch.exp(self[p + "A_log"]) * torch.nn.functional.softplus(self.linear(x, p + "a") + self[p + "dt_bias"]))
        S, out = x.new_zeros(H, D, V), []
        for t in range(T):
            S = S * g[t, :, None, None]
            u = beta[t, :, None] * (v[t] - (S * k[t, :, :, None]).sum(1))
            S = S + k[t, :, :, None] * u[:, None, :]
            out.append((S * q[t, :, :, None]).sum(1))
        o = self.norm(torch.stack(out), p + "norm") * silu(self.linear(x, p + "g")).view(T, H, V)
        return self.linear(o.reshape(T, H * V), p + "o")

    def differential(self, x, p, m):
        T, H, G, D, V = len(x), m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = (self.conv(self.linear(x, p + n) + self[p + n + ".b"], self[p + n + ".conv"]) for n in "qkv")
        q, k = (self.rotate(t.view(T, -1, D), m["rot"]["dims"], m["rot"]["base"]) for t in (q, k))
        lam = torch.exp((self[p + "lq1"] * self[p + "lk1"]).sum()) - torch.exp((self[p + "lq2"] * self[p + "lk2"]).sum()) + m["diff"]
        a = [self.attend(q[:, i::2], k[:, i::2], v.view(T, G, V), m["scale"], m["mask"]["size"], m["mask"]["keep_first"]) for i in (0, 1)]
        return self.linear((self.unit(a[0] - lam * a[1], 1e-6) * (1.0 - m["diff"])).reshape(T, H * V), p + "o")

    def dezudra(self, h, parts):
        for l, layer in enumerate(self.cfg["layers"]):
            p, mix = f"l{l}.", self.gated_delta if layer["type"] == "delta" else self.differential
            x = self.norm(h, p + "norm1")
            h = h + self.norm(torch.cat([mix(x[s], p + "mix.", layer["mixer"]) for s in parts]), p + "norm1b")
        return h, "final.norm", "head"

    def general_delta(self, x, p, m):
        T, H, D = len(x), m["heads"], m["dim"]
        r, k, v = (self.linear(x, p + n).view(T, H, D) for n in "rkv")
        inner = self.linear(torch.tanh(self.linear(x, p + "w1")), p + "w2") + self[p + "w0"]
        decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(inner)).view(T, H, D)
        a = torch.sigmoid(self.linear(x, p + "a") + self[p + "a.b"]).view(T, H, D)
        u = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        S, out = x.new_zeros(H, D, D), []
        for t in range(T):
            read = (S * u[t, :, :, None]).sum(1)
            S = S * decay[t, :, :, None] - (a[t] * u[t])[:, :, None] * read[:, None, :] + k[t, :, :, None] * v[t, :, None, :]
            out.append((S * r[t, :, :, None]).sum(1))
        y = self.unit(torch.stack(out), 1e-6).reshape(T, H * D) * self[p + "norm"]
        return self.linear(y * torch.sigmoid(self.linear(x, p + "g")), p + "o")

    def lightning(self, x, p, m):
        T, H, D = len(x), m["heads"], m["dim"]
        q, k, v = (torch.nn.functional.silu(self.linear(x, p + n)).view(T, H, -1) for n in "qkv")
        decay = torch.tensor(m["decay"], device="cuda", dtype=F64)[:, None, None]
        S, out = x.new_zeros(H, D, m["vdim"]), []
        for t in range(T):
            S = S * decay + k[t, :, :, None] * v[t, :, None, :]
            out.append((S * q[t, :, :, None]).sum(1))
        y = self.norm(torch.stack(out).reshape(T, -1), p + "norm")
        return self.linear(y * torch.sigmoid(self.linear(x, p + "g")), p + "o")

    def latent(self, x, p, m):
        T, H, D, r = len(x), m["heads"], m["dim"], m["rot_dim"]
        q, d = self.linear(x, p + "q").view(T, H, D + r), self.linear(x, p + "dkv")
        c = self.norm(d[:, :m["kv_rank"]], p + "dkv.norm")
        turn = lambda t: self.rotate_neighbours(t, r, m["rot"]["base"])
        key_rot = turn(d[:, None, m["kv_rank"]:]).expand(T, H, r)
        q = torch.cat([q[..., :D], turn(q[..., D:])], -1)
        k = torch.cat([self.linear(c, p + "uk").view(T, H, D), key_rot], -1)
        return self.linear(self.attend(q, k, self.linear(c, p + "uv").view(T, H, -1), m["scale"]).reshape(T, -1), p + "o")

    def bibevik(self, h, parts):
        mixers = {"general_delta": self.general_delta, "lightning": self.lightning, "latent_attention": self.latent}
        for l, layer in enumerate(self.cfg["layers"]):
            p, limit = f"l{l}.", layer["mlp"]["limit"]
            x = self.norm(h, p + "norm1")
            y = torch.cat([mixers[layer["type"]](x[s], p + "mix.", layer["mixer"]) for s in parts])
            g = (self.linear(x, p + "mlp.gate") + self[p + "mlp.gate.b"]).clamp(max=limit)
            u = (self.linear(x, p + "mlp.up") + self[p + "mlp.up.b"]).clamp(-limit, limit)
            h = h + y + self.linear(g * torch.sigmoid(1.702 * g) * (u + 1.0), p + "mlp.down") + self[p + "mlp.down.b"]
        return h, "final.norm", "head"

    def logits(self, tokens, wanted):
        """Logits at the wanted places (numbered through all sequences)."""
        starts = [0]
        for t in tokens:
            starts.append(starts[-1] + len(t))
        parts = [slice(a, b) for a, b in zip(starts, starts[1:])]
        ids = torch.tensor([t for s in tokens for t in s], device="cuda")
        qwen = self.case["model"] in ("a27b", "57b")
        h = self.w["model.embed_tokens.weight" if qwen else "embed"][ids].to(F64)
        h, norm, head = (self.qwen if qwen else getattr(self, self.case["model"]))(h, parts)
        return [self.linear(self.norm(h[torch.tensor([starts[i] + n for i, n in rows], device="cuda")], norm), head) for rows in wanted]


def exact(case, seed):
    tokens = _tokens(case, seed)
    if sum(len(t) for t in tokens) > 30000:  # (64 contexts, 16 of the largest model: too long in 64 bits)
        return None
    ends = [len(t) - case["new"] for t in tokens]
    last = lambda i: 1 if case["do"] in ("decode", "mixed") and i < case["requests"] else case["wanted"]
    wanted = [[(i, n) for i, end in enumerate(ends) for n in range(end - last(i), end)]]
    wanted += [[(i, end + k) for i, end in enumerate(ends)] for k in range(case["new"])]
    with torch.no_grad():
        out = _Plain(case, seed).logits(tokens, wanted)
    return out[0] if case["do"] in ("decode", "mixed") else out
