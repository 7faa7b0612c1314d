"""Mixture-of-experts feed-forward with an optional (sigmoid-gated) shared expert.

route -> group -> gate|up of the routed experts (+SwiGLU) -> down -> weighted
sum in slot order + shared expert (reference: MoeFfn::ForwardImpl,
src/model/moe_ffn.cc:158-367; kernels src/backends/cuda/ops/moe.cu).  Expert
weights are stacked at load: w13 [E, 2*mi, H] (gate rows, then up rows, per
expert) and w2 [E, H, mi] (reference: moe_ffn.h:25-34; stacking pattern
src/model/deepseek_v2.cc:515-542).  Router scores and the shared gate are
float32 from the product on.

Two options beside that: experts without a gate (`gated=False`: down(act(up x)) with act the square of relu, weights
w13 [E, mi, H]) and a router that chooses among groups (`groups`, `groups_keep`: the experts form equal groups of
neighbours, a group's score is its best expert's, and only experts of the best `groups_keep` groups can be chosen).
Further: `score` "sigmoid" (an expert's score is the sigmoid of its own logit, not the softmax over all),
`group_score` "top2" (a group's score is the sum of its two best experts'), and the activation "clamped_glu" with
`limit` (and `shared_limit` for the shared expert): g = min(gate, limit), u = clamp(up, -limit, limit),
g sigmoid(1.702 g) (u + 1).  `router_bias`: a learned number per expert joins its score before anything else (with
`renormalize` the weights are then the softmax over the chosen experts' biased scores alone).
"""
from __future__ import annotations

from typing import List, Optional

import torch

from .. import ops
from .base import FeedForward, LazyDelta, LazyNorm, ParamSpec, register_part
from .dense_mlp import stack_rows


# From here on the shared expert runs on a second stream beside the routed ones.  Below it a step of 24 layers
# waits for the host, which the two streams' hand-overs cost 21 us a layer (measured at the A2.7B shape, beside
# against one after the other: 8.1 against 7.0 ms at 256 tokens, 8.3 against 8.3 at 512, 9.0 against 9.8 at 768,
# 15.1 against 15.4 at 2,048).
SHARED_BESIDE_TOKENS = 512
# From this width on the LDS-staged expert products run in their wide form (256 weight rows per workgroup) and the
# shared expert stays on the main stream (a wide workgroup fills a compute unit's LDS, the library's kernels find
# no place beside it).  Measured, prompt portions at a width of 3,584 (64 experts of 2,560, 8 per token): 14.9 against
# 15.5 ms for a mixed step of 1,056 tokens and 8 layers, 2.86 against 3.03 s for 193,000 tokens of long prompts.
WIDE_TILES_WIDTH = 3072
# From this width on they do where no library product runs beside them: without a shared expert, or with it among the routed
# ones (below).  Both products at a width of 2,048 (60 experts of 1,408), us, narrow / wide: unevenly routed 512 tokens 209 /
# 191, 1,024 207 / 208, 2,048 272 / 247, 4,096 403 / 379; with the shared expert among them 64 tokens 170 / 166, 340 208 / 208, 768
# 255 / 234, 1,500 322 / 317, 2,048 412 / 380.
WIDE_TILES_ALONE_WIDTH = 2048
# ... and where both products of the narrow form would have so many workgroups, as the wide form has half as many, each with twice the
# work, and, without a shared expert's full tiles among them, so many rows a tile on average.  Wide against narrow, geometric means over 791
# shapes of 4 to 128 experts of 160 to 2,048 on widths of 2,048 and more: up to 512 workgroups 1.32, 1,024 1.11, 1,536 1.06, 2,048 1.06
# (eight experts of 768 on 2,048, 203 tokens of six, both products: 53 against 62 us), beyond without a shared expert with less than 32
# rows a tile 1.07, with more 0.99, with one 1.03 and 0.98 (64 tokens of 60 experts of 1,408, 8 layers, 2,574 us narrow, 2,541 wide).
WIDE_TILES_ALONE_WORKGROUPS = 2048
WIDE_TILES_ALONE_ROWS = 32
# The wide form's workgroups stay and take tile after tile (where the shapes allow it: `ops.moe_stays`) from so many tokens on.  Whole
# steps, us, a workgroup for each tile / staying: A2.7B shape, 8 layers, prompts of 48 tokens 1,367 / 1,429, 72 1,450 / 1,455, 100 1,587 /
# 1,543, 256 1,973 / 1,910, 768 2,775 / 2,647; 64 experts of 1,408 on 2,048 with two pieces, 8 layers, 72 1,487 / 1,541, 100 1,554 / 1,552,
# 192 1,832 / 1,734; 57B shape, 4 layers, portions of 48 2,880 / 2,883, 96 2,998 / 3,002, 128 3,113 / 3,092; 2 layers, 256 1,979 / 1,845.
STAY_TOKENS = 96
# ... as long as the weights of the first product are no more than so many MiB a compute unit, and so many more for each row that a tile
# has.  A tile of few rows waits for its weights alone, and one workgroup a tile has a stage more of them on its way: what that
# gains grows with the weights, while staying gains a tile's start and end.  Whole steps again, 100 | 256 | 384 | 768 tokens: 256
# experts of 2,048 on 4,096 (32 MiB; 4, 9, 13 and 27 rows a tile), 3 layers, 4,375 / 4,679 | 5,585 / 6,057 | 5,922 / 6,407 | 6,660 / 6,841
# and 1,200 tokens (42 rows) 7,245 / 7,275; 160 of 1,536 on 5,120 (19 MiB; 5, 13, 19, 38), 3 layers, 3,390 / 3,416 | 3,892 / 3,978 | 4,052 /
# 4,078 | 4,506 / 4,409; 128 of 1,536 on 4,096 (12 MiB; 7, 18, 27, 54), 4 layers, 2,842 / 2,833 | 3,332 / 3,321 | 3,622 / 3,543 | 4,044 /
# 3,942; 256 of 768 on 2,048 (6 MiB; 4, 9, 13, 27), 6 layers, 1,212 / 1,186 | 1,474 / 1,394 | 1,655 / 1,575 | 2,028 / 1,942.
STAY_MIB, STAY_MIB_A_ROW = 8.0, 0.625
# Between the few rows of a decoding step (where routed and shared experts already share a launch) and the portions
# from which the shared expert's library products run beside the routed experts, the shared expert is cut into
# pieces of the routed experts' width, which every token "chooses" with the shared gate's value as their weight:
# grouping, the two grouped products and the weighted sum then take it along, its weights stream at the rate of the
# big launches instead of through two library products of few rows and a launch for SwiGLU.  Needs a shared width
# that is a multiple of the experts' width; keeps the shared expert's weights a second time, in that layout.
# us of a whole prompt, without / with: A2.7B shape (8 layers) 300 tokens 2,672 / 2,430, 1,024 3,883 / 3,422; 57B shape (4 layers)
# 1,024 tokens 6,290 / 5,550, 1,500 7,522 / 7,263.
# Each piece's result is rounded before the sum adds them in float32: four (57B shape: eight) roundings of a half the size (a third)
# instead of one.
FOLD_SHARED_BELOW_TOKENS = 1536
# From there on, as far as the wide form goes, the shared expert's products are worked in the launches of the grouped ones as they
# are, each result one sum in 32 bits with one rounding.  A tile of the down product is then as long as those of all pieces, and
# worked first, so that it ends with the others as long as the pieces are few.  us of a whole prompt, by itself / in pieces / in the
# launches: A2.7B shape (8 layers) 1,536 tokens 4,090 / 4,185 / 4,110, 1,800 4,815 / 4,675 / 4,520, 2,112 5,175 / 5,105 / 4,915, 57B shape (4
# layers) 1,536 7,575 / 7,175 / 7,100, 2,048 9,135 / 9,025 / 8,810.  The line is eleven whole tiles of the wide form.
FOLD_SHARED_WHOLE_BELOW_TOKENS = 11 * ops.MOE_TILED_ROWS_WIDE + 1
FOLD_SHARED_WHOLE_PIECES = 8


class MoeFeedForward(FeedForward):
    graph_safe = True

    def __init__(self, hidden_size: int, num_experts: int, top_k: int, expert_width: int, shared_width: int = 0,
                 shared_gated: bool = True, renormalize: bool = False, routed_scale: float = 1.0,
                 init_std: float = 0.02, gated: bool = True, activation: Optional[str] = None, groups: int = 1,
                 groups_keep: int = 1, score: str = "softmax", group_score: str = "best", limit: float = 0.0,
                 shared_limit: Optional[float] = None, router_bias: bool = False):
        if not 0 < top_k <= num_experts:
            raise ValueError(f"top_k {top_k} must be between 1 and num_experts {num_experts}")
        if num_experts > 1024 or top_k > 32:
            raise ValueError("at most 1024 experts and top_k 32 are supported")
        self.hidden_size, self.num_experts, self.top_k = int(hidden_size), int(num_experts), int(top_k)
        self.expert_width, self.shared_width = int(expert_width), int(shared_width)
        self.shared_gated, self.renormalize = bool(shared_gated), bool(renormalize)
        self.routed_scale, self.init_std = float(routed_scale), float(init_std)
        self.gated = bool(gated)
        activation = activation or ("silu" if self.gated else "relu2")
        if (self.gated, activation) not in ((True, "silu"), (True, "clamped_glu"), (False, "relu2")):
            raise ValueError(f"experts {'with' if self.gated else 'without'} a gate and the activation {activation!r}: "
                             "a gate goes with silu or clamped_glu, no gate with relu2 (the square of relu)")
        if score not in ("softmax", "sigmoid") or group_score not in ("best", "top2"):
            raise ValueError(f"router scores {score!r} (softmax or sigmoid), group scores {group_score!r} (best or top2)")
        self.sigmoid_scores, self.group_top2 = score == "sigmoid", group_score == "top2"
        # the clamped activation's limits (0: the activation is silu(gate) * up)
        self.limit = float(limit) if activation == "clamped_glu" else 0.0
        self.shared_limit = self.limit if shared_limit is None or activation != "clamped_glu" else float(shared_limit)
        if activation == "clamped_glu" and (self.limit <= 0 or self.shared_limit <= 0):
            raise ValueError("the clamped activation needs a positive limit")
        if not self.gated and shared_width:
            raise ValueError("a shared expert needs gated experts")
        self.activation = activation
        # what the first grouped product does with its sums
        self.first_epilogue = ops.GATE_UP_SWIGLU if self.gated else ops.RELU_SQUARED
        self.groups, self.groups_keep = int(groups), int(groups_keep)
        if (self.groups < 1 or self.num_experts % self.groups or not 1 <= self.groups_keep <= self.groups
                or self.top_k > self.groups_keep * (self.num_experts // self.groups) or self.groups > 64):
            raise ValueError(f"{self.num_experts} experts in {groups} groups of which {groups_keep} are kept for "
                             f"top_k {self.top_k}: at most 64 equal groups, and the kept ones must hold top_k experts")
        self.wide_tiles = self.hidden_size >= WIDE_TILES_WIDTH
        # pieces of the routed experts' width that the shared expert is cut into for steps of middling size, or 0
        self.shared_pieces = self.shared_width // self.expert_width if (
            self.shared_width > 0 and self.shared_width % self.expert_width == 0
            and self.shared_width // self.expert_width <= 32 and self.shared_limit == self.limit) else 0
        self.w13_all = self.w2_all = None  # routed experts, then the shared expert's pieces
        self.router_bias = bool(router_bias)
        self.w_router = self.b_router = self.w13 = self.w2 = None
        self.w_shared_gate_up = self.w_shared_down = self.w_shared_gate = None

    def param_specs(self) -> List[ParamSpec]:
        H, mi, si, s = self.hidden_size, self.expert_width, self.shared_width, self.init_std
        specs = [ParamSpec("gate.weight", (self.num_experts, H), std=s)]
        if self.router_bias:
            specs.append(ParamSpec("gate.bias", (self.num_experts,), std=0.5))
        for e in range(self.num_experts):
            if self.gated:
                specs.append(ParamSpec(f"experts.{e}.gate_proj.weight", (mi, H), std=s))
            specs += [ParamSpec(f"experts.{e}.up_proj.weight", (mi, H), std=s),
                      ParamSpec(f"experts.{e}.down_proj.weight", (H, mi), std=s)]
        if si > 0:
            specs += [ParamSpec("shared_expert.gate_proj.weight", (si, H), std=s),
                      ParamSpec("shared_expert.up_proj.weight", (si, H), std=s),
                      ParamSpec("shared_expert.down_proj.weight", (H, si), std=s)]
            if self.shared_gated:
                specs.append(ParamSpec("shared_expert_gate.weight", (1, H), std=s))
        return specs

    def bind(self, tensors, rt) -> None:
        E = self.num_experts
        self.w_router = tensors["gate.weight"].contiguous()
        if self.router_bias:
            self.b_router = tensors["gate.bias"].to(torch.float32).contiguous()
        parts = []
        for e in range(E):
            if self.gated:
                parts.append(tensors[f"experts.{e}.gate_proj.weight"])
            parts.append(tensors[f"experts.{e}.up_proj.weight"])
        downs = [tensors[f"experts.{e}.down_proj.weight"] for e in range(E)]
        mi, S = self.expert_width, self.shared_pieces
        fold = S > 0 and self.gated and all(t.dtype == torch.bfloat16 for t in parts + downs) and all(
            tensors[f"shared_expert.{n}_proj.weight"].dtype == torch.bfloat16 for n in ("gate", "up", "down"))
        if fold:  # piece c of the shared expert: its gate rows, its up rows, and the columns of the down product
            for c in range(S):
                parts += [tensors["shared_expert.gate_proj.weight"][c * mi:(c + 1) * mi],
                          tensors["shared_expert.up_proj.weight"][c * mi:(c + 1) * mi]]
                downs.append(tensors["shared_expert.down_proj.weight"][:, c * mi:(c + 1) * mi])
        else:
            self.shared_pieces = S = 0
        self.w13_all = stack_rows(parts).view(E + S, (2 if self.gated else 1) * mi, self.hidden_size)
        self.w2_all = stack_rows(downs).view(E + S, self.hidden_size, mi)
        self.w13, self.w2 = self.w13_all[:E], self.w2_all[:E]
        if self.shared_width > 0:
            self.w_shared_gate_up = stack_rows([tensors["shared_expert.gate_proj.weight"],
                                                tensors["shared_expert.up_proj.weight"]])
            self.w_shared_down = tensors["shared_expert.down_proj.weight"].contiguous()
            if self.shared_gated:
                self.w_shared_gate = tensors["shared_expert_gate.weight"].contiguous()

    # -- the steps, separately callable so tests can look between them ----
    def route(self, ctx, x, always: int = 0):
        """`always`: the shared expert's pieces follow each token's chosen experts, with the shared gate's value (or
        1) as their weight."""
        rt, T, k = ctx.rt, x.shape[0], self.top_k + always
        topk_w = rt.empty((T, k), torch.float32)
        topk_e = rt.empty((T, k), torch.int32)
        gate = rt.empty((T,), torch.float32) if self.w_shared_gate is not None else None
        ops.moe_route(x, self.w_router, self.w_shared_gate, topk_w, topk_e, gate, self.renormalize, self.routed_scale,
                      always, self.groups, self.groups_keep, self.sigmoid_scores, self.group_top2, self.b_router)
        return topk_w, topk_e, gate

    def _tile_rows(self, ctx, x) -> int:
        """Rows per tile of the matrix-core product, or 0 where it does not take the shapes (then the plain one runs)."""
        piece = 16 // x.element_size()  # (rows are read 16 bytes at a time)
        ok = (self.w13.dtype == x.dtype and self.w2.dtype == x.dtype and self.hidden_size % piece == 0
              and self.expert_width % piece == 0 and (x.dtype == torch.bfloat16 or self._f32_fits(x)))
        if not ok:
            return 0
        # A decoding step, or few rows per expert: 16-row tiles, the weights streamed by every wavefront for itself.
        # From about three rows per expert on the LDS-staged kernel is faster (60 experts, 4 per token: 174 against
        # 173 us for both products at 48 tokens, 209 against 189 at 96, 316 against 195 at 256).  The float32 forms go by
        # the same line (33 tokens 345 against 334, 48 358 against 349, 96 411 against 371, 256 645 against 397).
        per_expert = x.shape[0] * self.top_k / self.num_experts
        if x.shape[0] <= ctx.rt.SKINNY_ROWS or per_expert <= 3:
            return 16
        if x.dtype == torch.float32:
            return ops.MOE_TILED_F32_ROWS
        wide = self.wide_tiles or (self._wide(x.shape[0]) and self._enough_for_wide(x.shape[0]))
        return ops.moe_tiled_rows(wide)

    def _enough_for_wide(self, tokens: int) -> bool:
        """Whether the LDS-staged products have the workgroups and the rows for their wide form, the shared expert's pieces among them."""
        rows = tokens * (self.top_k + self.shared_pieces)
        tiles = ops.moe_tiled_tiles(rows, self.num_experts + self.shared_pieces)
        columns = ops.moe_tiled_columns(self.expert_width, self.gated) + ops.moe_tiled_columns(self.hidden_size, False)
        return tiles * columns >= WIDE_TILES_ALONE_WORKGROUPS and (
            self.shared_pieces > 0 or rows >= WIDE_TILES_ALONE_ROWS * tiles)

    def _wide(self, tokens: int) -> bool:
        """Whether the width lets the LDS-staged products of this step take their wide form."""
        alone = self.shared_width == 0 or self._shared_rides_along(tokens) or self._shared_in_the_launches(tokens)
        return self.wide_tiles or (alone and self.hidden_size >= WIDE_TILES_ALONE_WIDTH)

    def _f32_fits(self, x) -> bool:
        """What the float32 products on the matrix cores ask for beside whole 16-byte pieces: rows on 16-byte boundaries
        and 32-bit offsets."""
        A = x.shape[0] * self.top_k
        return (x.data_ptr() % 16 == 0 and max(x.shape[0] * self.hidden_size, A * self.expert_width) < 1 << 31
                and (2 if self.gated else 1) * self.expert_width * self.hidden_size < 1 << 31
                and ops.moe_max_tiles(A, self.num_experts, 16) < 65536)

    def _staying_pays(self, tokens: int, assignments: int, experts: int) -> bool:
        """Whether the wide form's workgroups had better stay than be as many as tiles."""
        tiles = ops.moe_tiled_tiles(assignments, experts)
        weights = tiles * (4 if self.gated else 2) * self.expert_width * self.hidden_size / ops.MOE_TILED_ALONE
        return tokens >= STAY_TOKENS and weights <= (STAY_MIB + STAY_MIB_A_ROW * assignments / tiles) * 2 ** 20

    def dispatch(self, ctx, topk_e, tile_rows: int = 0, always: int = 0):
        rt, A, E = ctx.rt, topk_e.numel(), self.num_experts + always
        offsets = rt.empty((E + 1,), torch.int32)
        rows = rt.empty((A,), torch.int32)
        dest = rt.empty((A,), torch.int32)
        tile_map = queues = None
        if tile_rows:
            mt, T = ops.moe_max_tiles(A, E, tile_rows), topk_e.shape[0]
            n, second_rows = 2 * mt + 1, T if not always and self._shared_in_the_launches(T) else 0
            stays = (tile_rows == ops.MOE_TILED_ROWS_WIDE and self._staying_pays(T, A, E)
                     and ops.moe_stays(A, E, self.hidden_size, self.expert_width, second_rows, self.shared_width))
            # (the queues of the wide form's two products lie behind the map, on a boundary of eight bytes)
            tile_map = rt.empty((n + 1 + ops.moe_queues_size(mt) if stays else n,), torch.int32)
            queues = tile_map[n + 1:] if stays else None
        ops.moe_dispatch(topk_e, offsets, rows, dest, E, tile_rows, tile_map, queues)
        return offsets, rows, dest, tile_map

    def experts(self, ctx, x, offsets, rows, tile_map=None, tile_rows: int = 0, with_shared: bool = False, shared=None):
        """`with_shared`: the grouping holds the shared expert's pieces as further experts.  `shared` [T, hidden]: the shared
        expert's products go into the launches of the wide form and leave their results there."""
        rt, A = ctx.rt, rows.numel()
        w13, w2 = (self.w13_all, self.w2_all) if with_shared else (self.w13, self.w2)
        act = rt.empty((A, self.expert_width))
        y = rt.empty((A, self.hidden_size))
        if tile_rows == ops.MOE_TILED_F32_ROWS:  # a float32 run, more than a few rows per expert
            ops.moe_grouped_tiled_f32(x, w13, act, offsets, rows, tile_map, self.first_epilogue, self.limit)
            ops.moe_grouped_tiled_f32(act, w2, y, offsets, None, tile_map, False)
        elif tile_rows in (ops.MOE_TILED_ROWS, ops.MOE_TILED_ROWS_WIDE):  # many rows per expert: operands staged through LDS
            wide = tile_rows == ops.MOE_TILED_ROWS_WIDE
            # (a piece of the shared expert holds every token: its tiles are full, and the last ones of the map)
            each = -(-x.shape[0] // tile_rows)
            full = self.shared_pieces * each if with_shared else 0
            first = second = None
            if shared is not None:
                shared_act = rt.empty((x.shape[0], self.shared_width))
                first, second = (x, self.w_shared_gate_up, shared_act), (shared_act, self.w_shared_down, shared)
            n = 2 * ops.moe_max_tiles(A, w13.shape[0], tile_rows) + 2
            queues = tile_map[n:] if wide and tile_map.numel() > n else None  # (`dispatch`)
            ops.moe_grouped_tiled(x, w13, act, offsets, rows, tile_map, self.first_epilogue, wide, self.limit, full, each, first, queues, 0)
            ops.moe_grouped_tiled(act, w2, y, offsets, None, tile_map, False, wide, 0.0, full, each, second, queues, 1)
        elif tile_rows:
            # few rows: the weights are the traffic, the reduction is split over a workgroup's four wavefronts
            ops.moe_grouped_mfma(x, w13, act, offsets, rows, tile_map, tile_rows, self.first_epilogue, 4, self.limit)
            ops.moe_grouped_mfma(act, w2, y, offsets, None, tile_map, tile_rows, False, 4)
        else:
            ops.moe_grouped_plain(x, w13, act, offsets, rows, gate_up=self.first_epilogue, glu_limit=self.limit)
            ops.moe_grouped_plain(act, w2, y, offsets, None, gate_up=False)
        return y

    def _one_launch(self, ctx, x, tile_rows: int) -> bool:
        """Few tokens (decoding): routed and shared experts go into one launch per product."""
        return (tile_rows == 16 and self.shared_width > 0 and self.shared_width % (16 // x.element_size()) == 0
                and x.shape[0] <= ctx.rt.SKINNY_ROWS and self.w_shared_gate_up.dtype == x.dtype
                and self.w_shared_down.dtype == x.dtype
                and (x.dtype == torch.bfloat16 or self.w_shared_down.data_ptr() % 16 == 0))

    def experts_and_shared(self, ctx, x, offsets, rows, tile_map, tile_rows):
        rt, A, T = ctx.rt, rows.numel(), x.shape[0]
        act, sact = rt.empty((A, self.expert_width)), rt.empty((T, self.shared_width))
        ops.moe_grouped_dual(x, self.w13, act, offsets, rows, tile_map, tile_rows, x, self.w_shared_gate_up, sact, True,
                             self.limit, self.shared_limit)
        y, sout = rt.empty((A, self.hidden_size)), rt.empty((T, self.hidden_size))
        ops.moe_grouped_dual(act, self.w2, y, offsets, None, tile_map, tile_rows, sact, self.w_shared_down, sout, False)
        return y, sout

    def shared(self, ctx, x):
        rt = ctx.rt
        return rt.linear(rt.gated_linear(x, self.w_shared_gate_up, limit=self.shared_limit), self.w_shared_down)

    def route_and_dispatch(self, ctx, x, tile_rows: int, norm=None, always: int = 0):
        """`route` then `dispatch`; for the few tokens of a decoding step in one launch, and the norm before the
        feed-forward with them: `norm` = (h, delta, weight, eps, x), x still to be filled.  `always`: see `route`
        (the chosen experts are then the first `top_k` columns of what is returned)."""
        rt, T, k, E = ctx.rt, x.shape[0], self.top_k, self.num_experts
        if always or not self._routes_in_one_launch(T):
            assert norm is None
            topk_w, topk_e, gate = self.route(ctx, x, always)
            return (topk_w, topk_e, gate) + self.dispatch(ctx, topk_e, tile_rows, always)
        topk_w = rt.empty((T, k), torch.float32)
        topk_e = rt.empty((T, k), torch.int32)
        gate = rt.empty((T,), torch.float32) if self.w_shared_gate is not None else None
        offsets = rt.empty((E + 1,), torch.int32)
        rows = rt.empty((T * k,), torch.int32)
        dest = rt.empty((T * k,), torch.int32)
        tile_map = rt.empty((2 * ops.moe_max_tiles(T * k, E, tile_rows) + 1,), torch.int32) if tile_rows else None
        ops.moe_route_dispatch(None if norm else x, self.w_router, self.w_shared_gate, topk_w, topk_e, gate,
                               self.renormalize, self.routed_scale, offsets, rows, dest, tile_rows, tile_map, norm,
                               self.groups, self.groups_keep, self.sigmoid_scores, self.group_top2, self.b_router)
        return topk_w, topk_e, gate, offsets, rows, dest, tile_map

    def _routes_in_one_launch(self, tokens: int) -> bool:
        """Whether the router's scores, selection and grouping of this step fit the one launch for few tokens."""
        return ops.route_one_launch_fits(tokens, self.hidden_size, self.num_experts)

    def _shared_rides_along(self, tokens: int) -> bool:
        """Whether the shared expert is among the routed ones, in pieces, in a step of so many tokens: up to the line above, and
        as far as the grouped products' 32-bit places reach."""
        rows = tokens * (self.top_k + self.shared_pieces)
        return self.shared_pieces > 0 and tokens < FOLD_SHARED_BELOW_TOKENS and rows * self.expert_width < 1 << 31

    def _shared_in_the_launches(self, tokens: int) -> bool:
        """Whether the shared expert's products, whole, go into the grouped products' launches in a step of so many tokens."""
        return (0 < self.shared_pieces <= FOLD_SHARED_WHOLE_PIECES and self.hidden_size >= WIDE_TILES_ALONE_WIDTH
                and (self.w_shared_down is None or self.w_shared_down.data_ptr() % 16 == 0)
                and FOLD_SHARED_BELOW_TOKENS <= tokens < FOLD_SHARED_WHOLE_BELOW_TOKENS
                and max(tokens, 2 * self.hidden_size) * self.shared_width < 1 << 31)

    takes_lazy_norm = True

    def forward(self, ctx, x):
        norm = None
        if isinstance(x, LazyNorm):
            # a decoding step: the norm is applied by the router's kernel, which every token's row passes anyway
            rms = x.rms_operands()
            if rms is not None and self._routes_in_one_launch(x.h.shape[0]):
                lazy, x = x, ctx.rt.empty(tuple(x.h.shape))
                norm = (lazy.h, lazy.delta, rms[0], rms[1], x)
            else:
                x = x.materialize(ctx)
        tile_rows = self._tile_rows(ctx, x)
        one_launch = self._one_launch(ctx, x, tile_rows)
        if (tile_rows and not one_launch and norm is None and x.shape[0] > ctx.rt.SKINNY_ROWS
                and self._shared_rides_along(x.shape[0])):
            # a step of middling size: the shared expert rides along as pieces that every token chooses
            topk_w, _, _, offsets, rows, dest, tile_map = self.route_and_dispatch(ctx, x, tile_rows,
                                                                                  always=self.shared_pieces)
            y = self.experts(ctx, x, offsets, rows, tile_map, tile_rows, with_shared=True)
            return MoeSum(y, dest, topk_w, None, None, self.hidden_size)
        shared = join = None
        if tile_rows == ops.MOE_TILED_ROWS_WIDE and not one_launch and self._shared_in_the_launches(x.shape[0]):
            shared = ctx.rt.empty((x.shape[0], self.hidden_size))
            topk_w, _, gate, offsets, rows, dest, tile_map = self.route_and_dispatch(ctx, x, tile_rows, norm)
            y = self.experts(ctx, x, offsets, rows, tile_map, tile_rows, shared=shared)
            return MoeSum(y, dest, topk_w, shared, gate, self.hidden_size)
        if (not one_launch and self.shared_width > 0 and tile_rows == ops.MOE_TILED_ROWS
                and x.shape[0] >= SHARED_BESIDE_TOKENS and ctx.rt.can_run_beside()):
            # a prompt portion: the shared expert's library products are bound by the matrix cores, the routed
            # experts' kernels by memory, so the two run beside each other on two streams
            shared, join = ctx.rt.run_beside(lambda: self.shared(ctx, x))
        topk_w, topk_e, gate, offsets, rows, dest, tile_map = self.route_and_dispatch(ctx, x, tile_rows, norm)
        if one_launch:
            y, shared = self.experts_and_shared(ctx, x, offsets, rows, tile_map, tile_rows)
        else:
            y = self.experts(ctx, x, offsets, rows, tile_map, tile_rows)
            if join is not None:
                join()
            elif self.shared_width > 0:
                shared = self.shared(ctx, x)
        return MoeSum(y, dest, topk_w, shared, gate, self.hidden_size)


class MoeSum(LazyDelta):
    """sum_s topk_w[t, s] * y[dest[t, s]] + gate[t] * shared[t], formed by whoever consumes it."""

    def __init__(self, y, dest, topk_w, shared, gate, width):
        self.y, self.dest, self.topk_w, self.shared, self.gate, self.width = y, dest, topk_w, shared, gate, width

    def materialize(self, ctx):
        out = ctx.rt.empty((self.topk_w.shape[0], self.width))
        ops.moe_combine(self.y, self.dest, self.topk_w, self.shared, self.gate, out)
        return out

    norms_in_groups = True  # `add_rmsnorm` takes `groups`: the norm over equal runs of the width

    def add_rmsnorm(self, ctx, h, weight, eps, rows, out, groups: int = 1) -> bool:
        if self.width * 4 > 60 * 1024:
            return False
        ops.moe_combine_add_rmsnorm(h, self.y, self.dest, self.topk_w, self.shared, self.gate, weight, out, eps, rows,
                                    groups=groups)
        return True

    def add_normed_rmsnorm(self, ctx, h, sum_weight, sum_eps, weight, eps, rows, out) -> bool:
        """As `add_rmsnorm`, with the sum passing an RMS norm of its own before it is added."""
        if self.width * 4 > 60 * 1024 or out is None:
            return False
        ops.moe_combine_add_rmsnorm(h, self.y, self.dest, self.topk_w, self.shared, self.gate, weight, out, eps, rows,
                                    sum_weight=sum_weight, sum_eps=sum_eps)
        return True


register_part("feed_forward", "moe", MoeFeedForward)
