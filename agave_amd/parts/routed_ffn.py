"""A routed feed-forward: a mixture of gated experts with a shared expert.

The router's logits are a 32-bit product of the feed-forward's input with the router matrix (kept in
32-bit).  Scores are the softmax over all router outputs; the choice goes by score + correction among the
outputs of the best groups, the weights are the plain scores times a factor (see
``agave_amd.config.spec.RoutedFfnSpec``); or (``score="softmax_top"``) the largest logits plus a bias are chosen and
weighted by the softmax over the chosen alone.  Outputs past the experts with weights are identity experts:
their result is the input row.  The chosen experts' rows are summed with their weights, the shared
expert's row is added, times the sigmoid of a logit per token where it has a gate (the gate's vector rides along
as one more row of the router matrix, so its product costs no kernel).  A shared expert of the experts' own form is one of
the experts to the products where that pays (see ``merges``).

Nothing on the host depends on the choice: every launch has the same shape whatever the tokens are, so a
decode step is recorded into a graph like any other.
"""
from __future__ import annotations

import math
from typing import List

import torch

from ..config.spec import RoutedFfnSpec
from ..ops import kernels, routed
from ..weights.loader import TensorNeed
from .base import BuildEnv, register
from .ffn import GatedFfn


# Experts from which a shared expert of their form is one of them in every step (and its matrices are held with theirs alone).
MERGED_ALWAYS = 64


def merges(n: int, n_experts: int, top: int, ff: int, hidden: int) -> bool:
    """Whether a step of ``n`` tokens takes a shared expert as one of ``n_experts`` + 1 of ``ff`` inner rows and ``hidden`` columns, of
    which a token chooses ``top``: two products and their starts and ends less, unless the shared expert's tiles, which has every
    token, make a round of workgroups more (2 on a compute unit in tiles of 128 rows, 3 in tiles of 64).  us, a whole
    feed-forward (its pairs sorted, which up to 256 no longer are, some 7 us less on either side), with it among them and apart:
    16 of 2,048 by 2,048, 4 chosen, 1 token 49 and 57, 32 108 and 130, 64 136 and 124, 512
    179 and 205, 700 240 and 201 (38 tiles of 128, 608 workgroups, and 32, 512), 1,024 255 and 281, 3,001 500 and 536; 8 of 1,536 by
    1,536 64 tokens 70 and 82, 2,048 186 and 170; 32 of 1,024 by 2,048 6 tokens 72 and 81, 48 117 and 114, 700 192 and 203, 1,300 252 and
    224; 4 of 4,096 by 4,096 48 tokens 160 and 142, 100 170 and 200, 400 242 and 228.  Over 24 numbers of tokens from 33 to 6,000 and
    nine sizes of 4 to 24 experts the rule takes 0.94 of the time apart (1.01 of the better of both, 1.16 at the worst).  From 64
    experts on one more is little: 64 of 1,024 by 2,048 (where the sort of few pairs no longer takes all experts) 1 token 48 and
    52, 8 118 and 121, 400 249 and 266, 2,048 428 and 444; 256 of 512 by 2,048 8 143 and 150, 200 473 and 474, 4,096 872 and 859."""
    if n_experts >= MERGED_ALWAYS or n <= 32:
        return True

    def rounds(shared: int, side: int) -> int:
        """Rounds of the gate's workgroups, the experts' pairs off their average to one side by what chance makes of it where all
        experts are as likely; a round of the kernels of 16 rows is not one of these."""
        tm = routed.tile_plan(n * (top + shared), n_experts + shared, True, ff, hidden)[0]
        if tm == 16:
            return 0
        pairs = n * top / n_experts
        pairs += side * math.sqrt(pairs * (1.0 - top / n_experts))
        tiles = n_experts * math.ceil(pairs / tm) + shared * math.ceil(n / tm)
        return math.ceil(tiles * math.ceil(ff / tm) / (512 if tm == 128 else 768))
    apart = rounds(0, 1)
    return apart == 0 or rounds(1, -1) <= apart


class RoutedFfn:
    @staticmethod
    def kernel_libraries(spec, dtype):
        return ("routed_ffn",)

    def __init__(self, spec: RoutedFfnSpec, weights, env: BuildEnv):
        s = spec
        if s.activation not in kernels.GATE_ACTIVATIONS:
            raise ValueError(f"routed feed-forward: unsupported activation {s.activation!r}; known: {sorted(kernels.GATE_ACTIVATIONS)}")
        self.n_outputs = s.n_experts + s.n_identity
        if self.n_outputs < 1 or self.n_outputs > routed.MAX_OUTPUTS:
            raise ValueError(f"routed feed-forward: {self.n_outputs} router outputs (1 to {routed.MAX_OUTPUTS})")
        if s.groups < 1 or s.groups > 64 or self.n_outputs % s.groups:
            raise ValueError(f"routed feed-forward: {self.n_outputs} router outputs do not form {s.groups} equal groups (at most 64)")
        if not 1 <= s.keep_groups <= s.groups:
            raise ValueError(f"routed feed-forward: {s.keep_groups} of {s.groups} groups kept")
        if not 1 <= s.top <= s.keep_groups * (self.n_outputs // s.groups):
            raise ValueError(f"routed feed-forward: {s.top} experts chosen of {s.keep_groups * (self.n_outputs // s.groups)} that can be")
        if s.score not in ("softmax_all", "softmax_top", "sigmoid"):
            raise ValueError(f"routed feed-forward: unknown way of scoring {s.score!r} (softmax_all, softmax_top, sigmoid)")
        if s.group_top not in (1, 2) or (s.normalise and (s.top > 64 or s.score == "softmax_top")):
            raise ValueError("routed feed-forward: a group counts by its largest or its two largest scores; weights are divided "
                             "by their sum for at most 64 chosen experts")
        if s.score == "softmax_top" and (s.groups != 1 or s.top > 64 or s.n_identity):
            raise ValueError("routed feed-forward: the softmax over the chosen logits takes no groups, no identity experts "
                             "and at most 64 chosen")
        if s.shared_gate and s.shared is None:
            raise ValueError("routed feed-forward: a gate on the shared expert needs a shared expert")
        self.spec, self.env = spec, env
        self.act = kernels.GATE_ACTIVATIONS[s.activation]
        dev = env.device
        # the router stays 32-bit in both engines
        rows = [weights.get(s.router).to(torch.float32)]
        if s.shared_gate:
            rows.append(weights.get(s.shared_gate).to(torch.float32).view(1, s.hidden))
        self.router = torch.cat(rows, 0).contiguous().to(dev)
        # A shared expert of the experts' own form may be one more of them (the last), and every token's last pair: two products and
        # their starts and ends less, and 32-bit rows.  From MERGED_ALWAYS experts on its matrices are then held with theirs and
        # nowhere else, with fewer of them also in a feed-forward of its own.
        names = (s.shared.gate_proj, s.shared.up_proj, s.shared.down_proj) if s.shared is not None else ()
        self.shared_as_expert = bool(
            s.shared is not None and 0 < s.n_experts < routed.MAX_OUTPUTS and not s.n_identity and env.dtype == torch.bfloat16
            and s.hidden % 32 == 0 and s.intermediate % 32 == 0
            and (s.shared.hidden, s.shared.intermediate, s.shared.activation) == (s.hidden, s.intermediate, s.activation)
            and (s.shared.act_limit, s.shared.act_alpha) == (s.act_limit, s.act_alpha)
            and not (s.shared.gate_bias or s.shared.up_bias or s.shared.down_bias)
            and all(env.weight_dtype(weights.get(name).dtype) == torch.bfloat16 for name in names))
        self.correction = weights.get(s.correction).to(torch.float32).contiguous().to(dev) if s.correction else None

        def stack(which: str) -> torch.Tensor:
            mats = [weights.get(f"{s.expert_prefix}{i}.{which}") for i in range(s.n_experts)]
            if self.shared_as_expert:
                mats.append(weights.get(dict(zip((s.gate_name, s.up_name, s.down_name), names))[which]))
            return torch.stack([m.to(env.dtype) for m in mats]).contiguous().to(dev)     # [experts, out, in]
        # bfloat16 experts whose sizes are multiples of 32 are kept in the matrix cores' tile order (only that copy)
        self.tile_order = bool(s.n_experts) and env.dtype == torch.bfloat16 and s.hidden % 32 == 0 and s.intermediate % 32 == 0
        if s.n_experts:
            self.w_gate, self.w_up, self.w_down = stack(s.gate_name), stack(s.up_name), stack(s.down_name)
            if self.tile_order:
                self.w_gate, self.w_up, self.w_down = (routed.pack_expert_weights(w) for w in (self.w_gate, self.w_up, self.w_down))
        else:
            self.w_gate = self.w_up = self.w_down = None
        only_merged = self.shared_as_expert and s.n_experts >= MERGED_ALWAYS
        self.shared = GatedFfn(s.shared, weights, env) if s.shared is not None and not only_merged else None

    @staticmethod
    def tensor_needs(spec: RoutedFfnSpec) -> List[TensorNeed]:
        s = spec
        r = s.n_experts + s.n_identity
        needs = []
        for i in range(s.n_experts):
            p = f"{s.expert_prefix}{i}."
            needs += [TensorNeed(p + s.gate_name, (s.intermediate, s.hidden)), TensorNeed(p + s.up_name, (s.intermediate, s.hidden)),
                      TensorNeed(p + s.down_name, (s.hidden, s.intermediate))]
        needs.append(TensorNeed(s.router, (r, s.hidden)))
        if s.correction:
            needs.append(TensorNeed(s.correction, (r,)))
        if s.shared is not None:
            needs += GatedFfn.tensor_needs(s.shared)
        if s.shared_gate:
            needs.append(TensorNeed(s.shared_gate, (1, s.hidden)))
        return needs

    def forward(self, x: torch.Tensor, step) -> torch.Tensor:
        y = self.forward_pending(x, step)
        return y.rows() if isinstance(y, routed.RoutedRows) else y

    def forward_pending(self, x: torch.Tensor, step):
        """The result with its pairs' rows not added up yet (:class:`agave_amd.ops.routed.RoutedRows`), for a block whose next norm
        may do that; plain rows where some of the experts are identity experts, whose result is ``x``."""
        s, ws = self.spec, self.env.workspace
        n, r, top = x.shape[0], self.n_outputs, s.top
        merged = self.shared_as_expert and (self.shared is None or merges(n, s.n_experts, top, s.intermediate, s.hidden))
        experts, pairs = s.n_experts + merged, top + merged
        choice = ws.get("router_choice", n, pairs, torch.int32)
        weight = ws.get("router_weight", n, pairs, torch.float32)
        # the router's 32-bit product and the choice in one kernel
        shared_gate = ws.get("router_shared_gate", n, 1, torch.float32) if s.shared_gate and not merged else None
        routed.route_rows(x, self.router, self.correction, s.groups, s.keep_groups, top, s.route_scale, choice, weight,
                          softmax_top=s.score == "softmax_top", extra_out=shared_gate, sigmoid=s.score == "sigmoid",
                          group_top=s.group_top, normalise=s.normalise, shared_expert=s.n_experts if merged else None,
                          shared_gate=bool(merged and s.shared_gate))
        y = place = None
        if self.tile_order and not routed.mfma_ok(x, s.intermediate):
            raise ValueError("routed feed-forward: its experts are kept in tile order, which takes aligned bfloat16 rows")
        if s.n_experts and self.w_gate.dtype == torch.bfloat16 and routed.mfma_ok(x, s.intermediate):
            tm, tiles, cap = routed.tile_plan(n * pairs, experts, self.tile_order, s.intermediate, s.hidden)
            if self.tile_order and tm == 16 and routed.chosen_takes(n * pairs, experts, s.intermediate, s.hidden):
                # few pairs: the products find their rows from the choices themselves
                act_rows = ws.get("expert_act", n * pairs, s.intermediate, x.dtype)
                y = ws.get("expert_rows", n * pairs, s.hidden, torch.float32)
                routed.experts_chosen(x, choice.view(-1), self.w_gate, self.w_up, self.w_down, act_rows, y, pairs, self.act,
                                      s.act_limit, s.act_alpha)
            else:
                # the pairs sorted by expert on the device, then the experts' products tile by tile on the matrix cores
                place = ws.get("expert_place", n * pairs, 1, torch.int32).view(-1)
                sorted_pair = ws.get(f"expert_sorted{tm}", cap, 1, torch.int32).view(-1)
                tile_expert = ws.get(f"expert_tiles{tm}", tiles, 1, torch.int32).view(-1)
                routed.route_sort(choice.view(-1), experts, tm, tiles, place, sorted_pair, tile_expert)
                act_rows = ws.get("expert_act", cap, s.intermediate, x.dtype)
                y = ws.get("expert_rows", cap, s.hidden, torch.float32)
                routed.experts_mfma(x, sorted_pair, tile_expert, self.w_gate, self.w_up, self.w_down, act_rows, y, tm, tiles, pairs,
                                    self.act, tile_order=self.tile_order, p0=s.act_limit, p1=s.act_alpha)
        elif s.n_experts:
            act_rows = ws.get("expert_act", n * top, s.intermediate, x.dtype)
            y = ws.get("expert_rows", n * top, s.hidden, torch.float32)
            routed.experts_plain(x, choice.view(-1), self.w_gate, self.w_up, self.w_down, act_rows, y, top, self.act,
                                 s.act_limit, s.act_alpha)
        shared = self.shared.forward(x, step, slices_ok=False, tag="shared_ffn") if self.shared is not None and not merged else None
        out = ws.get("routed_out", n, s.hidden, x.dtype)
        pending = routed.RoutedRows(y, place, choice.view(-1), weight.view(-1), x, shared, out, pairs, experts,
                                    shared_gate.view(-1) if shared_gate is not None else None)
        return pending.rows() if s.n_identity or y is None else pending


register("ffn", "routed", RoutedFfn)
