"""Differential attention over the paged cache: every head has two score maps over one set of values, and its
result is the first map's minus lambda times the second's.

    q|k|v   = x . [Wq; Wk; Wv]^T + bias           q: heads x [map 0, map 1] x dim, k: kv_heads x [map 0, map 1] x dim,
                                                  v: kv_heads x vdim
    q, k, v = short_conv(.)                       causal, per channel, continued from the request's last inputs
    q, k    = rotated (the position encoding's part of every map)
    a_m     = softmax_j(q_m . k_m[j] * scale) v[j]    over the keys the query sees: j <= i and
                                                      (i - j < window or j < keep_first); window 0: all
    lambda  = exp(lq1 . lk1) - exp(lq2 . lk2) + diff  one number for the layer
    o       = a_0 - lambda a_1;  o / rms(o) * (1 - diff)           rms over a head's vdim, no weight
    y       = concat(o) . Wo^T

The cache keeps the rotated keys of both maps (2 kv_heads "heads" of dim) and the values (kv_heads of vdim,
transposed within a page); with a window the pages that it has passed go back, except those of the kept first
tokens.  The short convolution's last inputs live in the request's state slot.  Scores, softmax, the difference
and the norm are float32 in every run.
"""
from __future__ import annotations

import math
from typing import List, Optional

import numpy as np
import torch

from .. import ops
from ..config.spec import PartSpec
from .attention import MIN_KEYS_PER_SPLIT, PREFILL_MIN_ROWS, QUERY_TILE, WAVES_WANTED, _tiles_of, plan_tiles
from .base import CacheArray, CacheNeed, Mixer, ParamSpec, StateNeed, build_part, register_part
from .dense_mlp import stack_rows
from .short_conv import ShortConv


# A step that brings some request several tokens goes through the kernel that shares keys and values through LDS, or through the
# wavefront-level one, which cuts keys into slices where a step has few tiles.  A workgroup of the former (a tile of up to 64
# queries of a head) walks all of its keys however few queries it has, so which is the quicker goes by the rounds of 32 keys of
# the longest tile and of all tiles together (`portion_plan`).  The estimates are fitted to 2,776 steps of 0 to 64 single tokens
# on 100 to 4,000 keys beside portions of 2 to 700 on up to 3,000, 8 to 32 heads, maps and values of 64 and 128: the chosen kernel
# is 0.6 % from the quicker one on average (the LDS one always 49 %, the other 21 %).  us, wavefront-level / LDS, 16 heads:
# prompts of 611 and 1,437 with a window of 1,024 105 / 48, eight of 200 37 / 16; 64 tokens on 384 keys 16.3 / 18.6; 64 beside 32
# single tokens on 1,000 keys, the 64 a prompt of their own 68 / 52, on 1,500 68 / 80; beside sixteen on 2,000 64 / 90.  Where
# every request brings fewer than sixteen the wavefronts' rounds took a fifth less: sixteen of 5 tokens on 1,000 keys, values of
# 128, 38 / 51, forty on 600 45 / 56; sixty-four of 10 on 10 18 / 15.
# Single tokens on more than 2,048 keys go to a launch of their own, in slices, in one LDS launch / two: 1,200 tokens beside
# sixteen single ones on 1,500, 2,000, 3,000 and 30,000 89 / 84, 106 / 101, 142 / 107 and 1,141 / 306, beside four on 2,000 and
# 3,000 88 / 90 and 123 / 94.
PREFILL_TILE = 64
PREFILL_MAX_FEW_KEYS = 2048


class DifferentialAttention(Mixer):
    graph_safe = True  # every launch reads the step's device arrays only

    def __init__(self, hidden_size: int, num_heads: int, num_kv_heads: int, head_dim: int, value_dim: int,
                 diff: float, conv_taps: int = 1, scale: Optional[float] = None, window: int = 0, keep_first: int = 0,
                 norm_eps: float = 1e-6, position: Optional[PartSpec] = None, init_std: float = 0.02):
        if num_heads % num_kv_heads:
            raise ValueError(f"num_heads {num_heads} is not a multiple of num_kv_heads {num_kv_heads}")
        if not 0 < head_dim <= 256 or not 0 < value_dim <= 256:
            raise ValueError(f"head_dim {head_dim} and value_dim {value_dim} must be between 1 and 256")
        if window < 0 or keep_first < 0:
            raise ValueError("window and keep_first must not be negative")
        self.hidden_size, self.num_heads, self.num_kv_heads = int(hidden_size), int(num_heads), int(num_kv_heads)
        self.head_dim, self.value_dim = int(head_dim), int(value_dim)
        self.diff, self.norm_eps, self.init_std = float(diff), float(norm_eps), float(init_std)
        self.scale = float(scale) if scale is not None else self.head_dim ** -0.5
        self.window, self.keep_first = int(window), int(keep_first) if window > 0 else 0
        self.position = build_part("position", position) if position is not None else None
        if self.position is not None:
            dims = int(getattr(self.position, "rotary_dim", 0))
            if getattr(self.position, "begin", 0) != 0 or dims <= 0 or dims % 2 or dims > self.head_dim:
                raise ValueError(f"the position encoding must rotate the first {dims} elements of maps of "
                                 f"{self.head_dim}: an even number within the map, from its start")
        self.q_dim, self.k_dim = 2 * self.num_heads * self.head_dim, 2 * self.num_kv_heads * self.head_dim
        self.v_dim, self.o_dim = self.num_kv_heads * self.value_dim, self.num_heads * self.value_dim
        self.conv = ShortConv(self.q_dim, self.k_dim, self.v_dim, self.head_dim, self.value_dim, conv_taps)
        self.w_qkv = self.b_qkv = self.w_out = None
        self.lam = 0.0
        self.plan_key = ("attention_diff_portions", self.num_heads, self.num_kv_heads, self.head_dim, self.value_dim, self.window,
                         self.keep_first)

    def cache_need(self) -> CacheNeed:
        return CacheNeed((CacheArray("k", 2 * self.num_kv_heads, self.head_dim),
                          CacheArray("v", self.num_kv_heads, self.value_dim, transposed=True)),
                         self.window, self.keep_first)

    def state_need(self) -> StateNeed:
        return StateNeed((max(1, self.conv.state_floats),), "float32")

    def subparts(self):
        return [self.position]

    def param_specs(self) -> List[ParamSpec]:
        W, s, D = self.hidden_size, self.init_std, self.head_dim
        return [ParamSpec("q.weight", (self.q_dim, W), std=s), ParamSpec("k.weight", (self.k_dim, W), std=s),
                ParamSpec("v.weight", (self.v_dim, W), std=s), ParamSpec("q.bias", (self.q_dim,), std=s),
                ParamSpec("k.bias", (self.k_dim,), std=s), ParamSpec("v.bias", (self.v_dim,), std=s),
                ParamSpec("lq1", (D,), std=0.1), ParamSpec("lk1", (D,), std=0.1), ParamSpec("lq2", (D,), std=0.1),
                ParamSpec("lk2", (D,), std=0.1), ParamSpec("o.weight", (W, self.o_dim), std=s)] + self.conv.param_specs()

    def bind(self, tensors, rt) -> None:
        self.w_qkv = stack_rows([tensors[f"{n}.weight"] for n in "qkv"])
        self.b_qkv = stack_rows([tensors[f"{n}.bias"] for n in "qkv"])
        self.w_out = tensors["o.weight"].contiguous()
        self.conv.bind(tensors, bias=self.b_qkv)
        dot = lambda a, b: float((tensors[a].double() * tensors[b].double()).sum().item())
        self.lam = math.exp(dot("lq1", "lk1")) - math.exp(dot("lq2", "lk2")) + self.diff
        if self.position is not None:
            self.position.bind({}, rt)

    def forward(self, ctx, x, cache):
        rt, T = ctx.rt, x.shape[0]
        table = self.position.prepare(ctx) if self.position is not None else None
        proj = rt.linear(x, self.w_qkv)
        q = rt.empty((T, self.num_heads, 2, self.head_dim))
        if cache.writes:
            self.conv.apply(ctx, proj, cache.state, q, cache.k, cache.v, slots=ctx.slots[cache.group], cos_sin=table)
        else:  # the keys and values are another execution's: only the queries are wanted
            self.conv.apply(ctx, proj, cache.state, q, rt.empty((T, self.k_dim)), rt.empty((T, self.v_dim)),
                            cos_sin=table)
        out = rt.empty((T, self.num_heads, self.value_dim))
        self.attend(ctx, q, cache, out)
        return rt.linear(out.view(T, self.o_dim), self.w_out)

    def capture_plan(self, ctx, requests: int, longest: int) -> None:
        """The query tiles of a step of one token per request never change (tile i = request i, row i, one query);
        the slices of the keys follow from `longest`.  (The same plan, under the same key, as plain attention's.)"""
        key = ("attention_tiles_host", QUERY_TILE)
        if key not in ctx.memo:
            every = np.arange(requests, dtype=np.int32)
            tiles = ops.upload(np.stack([every, every, np.ones_like(every)]), ctx.rt.device)
            ctx.memo[key] = (tiles, requests, longest)

    def key_slices(self, units: int, longest: int) -> int:
        """Into how many slices each tile's keys are cut: enough wavefronts for the machine, no slice shorter than
        MIN_KEYS_PER_SPLIT, a power of two (few distinct values, few captured graphs), 64 at most."""
        span = min(longest, self.window + self.keep_first + QUERY_TILE + 32) if self.window > 0 else longest
        n = 1 if units >= WAVES_WANTED else max(1, min(WAVES_WANTED // max(1, units), -(-span // MIN_KEYS_PER_SPLIT), 64))
        return 1 << (n.bit_length() - 1)

    def portion_plan(self, ctx):
        """Which tiles the LDS-sharing kernel takes in a step that brings some request several tokens, or None if the
        wavefront-level kernel takes the step: (tiles, few), few = (rows, tiles, positions, slices, grouped) for a launch of the
        latter that serves the requests of few tokens by themselves, or None."""
        key = self.plan_key
        if key in ctx.memo:
            return ctx.memo[key]
        tiles, _, longest = plan_tiles(ctx, PREFILL_TILE)
        reach = self.window + self.keep_first if self.window > 0 else longest
        H, capped = self.num_heads, reach / 32 + 1
        q_start = ctx.host.q_start.tolist()
        shared = own = of_queries = few = 0  # rounds of all tiles of either kernel, the latter's tiles, requests of few tokens
        keys = most_new = 0                  # the longest context of those, the most tokens of a request
        for start, end, length in zip(q_start, q_start[1:], ctx.host.seq_lens.tolist()):
            n = end - start
            rounds = (2 * length - n) / 64  # of a tile on average
            rounds = 1 + (rounds if rounds < capped else capped)
            tiles16 = (n + 15) // 16
            shared += (n + 63) // 64 * rounds
            own += tiles16 * rounds
            of_queries += tiles16
            most_new = max(most_new, n)
            if 0 < n < PREFILL_MIN_ROWS:
                few += 1
                keys = max(keys, length)
        most = min(longest, reach + PREFILL_TILE) / 32
        slices = self.key_slices(of_queries * 2 * H, longest)
        wide = self.head_dim + self.value_dim
        through_lds = 9.0 + max(most * (0.64 + 0.0027 * wide), 1.7e-5 * wide * shared * H)
        own *= 2e-5 if most_new >= PREFILL_MIN_ROWS else 1.6e-5
        wavefronts = 9.1 + max(most / slices * (1.28 + 0.003 * wide), wide * own * H) + 2e-4 * ctx.num_tokens * H * slices
        plan = None
        if through_lds < wavefronts:
            plan = (tiles, None) if not few or min(keys, reach) <= PREFILL_MAX_FEW_KEYS else self._few_by_themselves(ctx, keys)
        ctx.memo[key] = plan
        return plan

    def _few_by_themselves(self, ctx, keys: int):
        """`portion_plan` with a launch of their own for the requests of few tokens (keys: the longest context among them): their
        rows are put side by side, since slices are merged for all rows of a launch."""
        q_start = ctx.host.q_start.astype(np.int64)
        n = q_start[1:] - q_start[:-1]
        few = np.flatnonzero((n > 0) & (n < PREFILL_MIN_ROWS))
        to_dev = lambda a: ops.upload(a, ctx.rt.device)
        grouped = 2 <= self.num_heads // self.num_kv_heads <= 16
        own = _tiles_of(n[few], np.cumsum(n[few]) - n[few], few, 1 if grouped else QUERY_TILE)
        rows = to_dev(np.concatenate([np.arange(q_start[i], q_start[i + 1]) for i in few]))
        slices = self.key_slices(own.shape[1] * 2 * (self.num_kv_heads if grouped else self.num_heads), keys)
        many = np.flatnonzero(n >= PREFILL_MIN_ROWS)
        return (to_dev(_tiles_of(n[many], q_start[many], many, PREFILL_TILE)),
                (rows, to_dev(own), ctx.positions.index_select(0, rows), slices, grouped))

    def attend(self, ctx, q, cache, out) -> None:
        """bfloat16 with heads and pages that the matrix-core kernels are built for: those, prompt portions in tiles of 64
        queries through LDS or, with the few tokens beside them, in tiles of up to 16 queries of a request, a (head, map) pair
        per wavefront (one token per request: the query heads of a key/value head side by side); else the plain one."""
        page_size = cache.k.shape[2]
        plan = None
        if (q.dtype == torch.bfloat16 and not ctx.one_token_each
                and ops.attention_diff_prefill_fits(self.head_dim, self.value_dim, page_size)):
            plan = self.portion_plan(ctx)
        if plan is not None:
            tiles, few = plan
            ops.attention_diff_prefill(q, cache.k, cache.v, ctx.block_tables[cache.group], tiles, ctx.positions, out,
                                       self.scale, self.window, self.keep_first, self.lam, self.norm_eps, 1.0 - self.diff)
            if few is not None:
                rows, tiles, positions, n_splits, grouped = few
                own = q.index_select(0, rows)
                result = ctx.rt.empty((rows.numel(), self.num_heads, self.value_dim))
                self._attend_wavefronts(ctx, own, cache, result, tiles, positions, n_splits, grouped)
                out.index_copy_(0, rows, result)
            return
        if q.dtype == torch.bfloat16 and ops.attention_diff_mfma_fits(self.head_dim, self.value_dim, page_size):
            tiles, n_tiles, longest = plan_tiles(ctx, QUERY_TILE)
            group = self.num_heads // self.num_kv_heads
            grouped = ctx.one_token_each and 2 <= group <= 16
            n_splits = self.key_slices(n_tiles * 2 * (self.num_kv_heads if grouped else self.num_heads), longest)
            self._attend_wavefronts(ctx, q, cache, out, tiles, ctx.positions, n_splits, grouped)
            return
        ops.attention_diff_plain(q, cache.k, cache.v, ctx.block_tables[cache.group], ctx.seq_of_token, ctx.positions,
                                 out, self.scale, self.window, self.keep_first, self.lam, self.norm_eps,
                                 1.0 - self.diff)

    def _attend_wavefronts(self, ctx, q, cache, out, tiles, positions, n_splits: int, grouped: bool) -> None:
        work = ctx.rt.empty((q.shape[0] * self.num_heads * 2 * n_splits * (self.value_dim + 2),), torch.float32)
        ops.attention_diff_mfma(q, cache.k, cache.v, ctx.block_tables[cache.group], tiles, positions, out, n_splits, work,
                                self.scale, self.window, self.keep_first, self.lam, self.norm_eps, 1.0 - self.diff,
                                grouped=grouped)


register_part("mixer", "differential_attention", DifferentialAttention)
