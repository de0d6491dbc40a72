"""A routed feed-forward: a mixture of small feed-forward layers (experts) of
which every token uses a few.

Router: z = Wr n in float32; scores s = softmax(z) over all router outputs;
the `top` outputs with the largest s + correction are chosen (the correction
moves the choice only) and their weights are their scores s, as they are, not
renormalized. The first `experts` router outputs are real experts,
y = Wdown act(Wup n) without biases; the last `identity` outputs stand for
experts that pass their input through. The result is the weighted sum of the
chosen experts' outputs, added in the order of the choice.

Parameters: width, hidden (an expert's), experts, identity, top, activation
("relu2": the square of max(z, 0); "swiglu": a gated expert, y = Wdown
(silu(Wgate n) * (Wup n)), whose gate matrix is named by `expert_gate`;
"clamped_glu": a gated expert whose unit has bounds, g sigmoid(alpha g) (u + 1)
with g = min(Wgate n, limit) and u = clamp(Wup n, -limit, limit), parameters
`limit` and `alpha`),
scoring ("softmax" over all router outputs, "sigmoid" of each output by
itself, or "chosen": the outputs themselves choose, and the weights are the
softmax over the chosen outputs alone), weigh ("output": a chosen expert's result is multiplied by its
weight; "input": the expert reads its input times its weight and the results
are added as they are), `group_count` and `group_keep` (the router outputs form
group_count equal groups of neighbours; a group's score is the sum of its two
largest score + correction, and only outputs of the group_keep best groups can
be chosen: an output of another group never is, however low the scores
inside the kept groups lie), `normalize` (the
chosen scores are divided by their sum + 1e-20), `route_scale` (a factor on the
weights), `shared` (the PartSpec of a feed-forward that every token uses; its
result is added, multiplied by sigmoid(Wsg n), one number a token, with Wsg the
tensor `shared_gate`; with `shared_gate` None it is added as it is), and the
tensors' names: `router`, `router_bias` (None: no bias on the router's outputs),
`correction` (None: no correction), `expert_up` / `expert_down` as patterns with `{e}` for the
expert's number.

A shared expert that is added as it is, of the experts' form and about their size,
is run as one expert more, which every token uses.

The experts' matrices lie stacked, [experts, out, in]. A step sorts its (token,
choice) entries by expert on the device and runs the two products over tiles of
one expert's rows each; the grids are sized by a bound the host knows, so
nothing comes back to the host and a step of this part can be captured.
"""
from __future__ import annotations

from typing import Dict, Optional

import torch

from ..config.plan import PartSpec
from ..kernels import ops
from ..weights.loader import TensorDecl
from .base import Declared, RouterRide, RowsToCombine, StepContext
from .linear import Linear, place_matrix, place_projection, place_vector
from .registry import part_class, register_part


GATED = ("swiglu", "clamped_glu")      # activations of experts with a gate matrix beside the way up


class RoutedExperts:
    role = "feed_forward"
    graph_safe = True     # launches kernels only: a step made of such parts can be captured

    @staticmethod
    def _names(spec: PartSpec) -> Dict[str, str]:
        names = dict(router="router", router_bias=None, correction="correction", expert_up="e{e}.up", expert_down="e{e}.down",
                     expert_gate="e{e}.gate", shared_gate="shared.sg")
        names.update(spec.get("names") or {})
        return {k: (None if v is None else f"{spec.prefix}.{v}") for k, v in names.items()}

    @classmethod
    def declare(cls, spec: PartSpec) -> Declared:
        n = cls._names(spec)
        E, F, X, I = spec["width"], spec["hidden"], spec["experts"], spec.get("identity", 0)
        out: Declared = {n["router"]: (TensorDecl((X + I, E)), "matrix")}
        for bias in ("correction", "router_bias"):
            if n[bias] is not None:
                out[n[bias]] = (TensorDecl((X + I,), "vector"), "bias")
        for e in range(X):
            if spec.get("activation", "relu2") in GATED:
                out[n["expert_gate"].format(e=e)] = (TensorDecl((F, E)), "matrix")
            out[n["expert_up"].format(e=e)] = (TensorDecl((F, E)), "matrix")
            out[n["expert_down"].format(e=e)] = (TensorDecl((E, F)), "matrix")
        if spec.get("shared") is not None:
            out.update(part_class("feed_forward", spec["shared"].kind).declare(spec["shared"]))
            if n["shared_gate"] is not None:
                out[n["shared_gate"]] = (TensorDecl((1, E)), "matrix")
        return out

    def __init__(self, spec: PartSpec, tensors: Dict[str, torch.Tensor], device: torch.device,
                 engine_dtype: torch.dtype):
        n = self._names(spec)
        self.width, self.hidden = spec["width"], spec["hidden"]
        self.experts, self.identity, self.top = spec["experts"], int(spec.get("identity", 0)), spec["top"]
        self.activation = spec.get("activation", "relu2")
        self.gated = self.activation in GATED
        self.alpha = 1.0
        limit = 0.0
        if self.activation == "clamped_glu":
            limit, self.alpha = float(spec["limit"]), float(spec.get("alpha", 1.702))
            if not limit > 0:
                raise ValueError(f"the bound of a clamped unit is positive, got {limit}")
        if not self.gated and (self.activation not in ops.MOE_EPILOGUES or self.activation in (None, "none")):
            raise ValueError(f"the experts' activation {self.activation!r} is not one the product's epilogue knows")
        self.scoring = spec.get("scoring", "softmax")
        if self.scoring not in ops.MOE_SCORINGS:
            raise ValueError(f"the router's scoring {self.scoring!r} is none of {sorted(ops.MOE_SCORINGS)}")
        if self.scoring == "chosen" and spec.get("normalize"):
            raise ValueError("a softmax over the chosen outputs is normalized already")
        self.weigh = spec.get("weigh", "output")
        if self.weigh not in ("output", "input"):
            raise ValueError(f"weigh is 'output' or 'input', got {self.weigh!r}")
        if self.weigh == "input" and (not self.gated or self.identity):
            # w act(W n) = act(W (w n)) holds for no activation here but the gated one's kernel, which takes w itself
            raise ValueError("experts that read their input times their weight are the gated ones, without pass-through experts")
        if not 1 <= self.top <= self.experts + self.identity:
            raise ValueError(f"{self.top} of {self.experts + self.identity} experts cannot be chosen")
        # bfloat16 x bfloat16 products are exact in float32 and the sums are float32: the router runs in 32 bits
        # on the matrix cores too; its input is the norm's output in the engine's dtype
        self.n_router = self.experts + self.identity
        self.group_count, self.group_keep = int(spec.get("group_count") or 1), int(spec.get("group_keep") or 1)
        if self.group_count > 1 and (self.n_router % self.group_count or not 1 <= self.group_keep <= self.group_count
                                     or self.group_keep * (self.n_router // self.group_count) < self.top):
            raise ValueError(f"{self.n_router} router outputs in {self.group_count} groups of which {self.group_keep} "
                             f"stay cannot give {self.top} choices")
        self.normalize, self.route_scale = bool(spec.get("normalize")), float(spec.get("route_scale", 1.0))
        router = tensors[n["router"]]
        self.shared, self.shared_gated = None, n["shared_gate"] is not None
        bias = None if n["router_bias"] is None else tensors[n["router_bias"]].to(torch.float32)
        shared = spec.get("shared")
        # a shared expert of the experts' own form and about their size is one of them that every token uses
        self.always = int(shared is not None and self._joins_experts(spec, shared))
        if shared is not None and not self.always:
            if shared.get("scratch_tag") is None:
                raise ValueError("a feed-forward inside this one keeps its scratch under a tag of its own (scratch_tag)")
            self.shared = part_class("feed_forward", shared.kind)(shared, tensors, device, engine_dtype)
        if self.shared is not None and self.shared_gated:
            # the shared expert's gate is one more row of the router's matrix: the same dot products, one launch
            gate = tensors[n["shared_gate"]].reshape(1, self.width)
            if gate.dtype != router.dtype:
                router, gate = router.to(torch.float32), gate.to(torch.float32)
            router = torch.cat([router, gate], dim=0)
            bias = None if bias is None else torch.cat([bias, bias.new_zeros(1)])
        self.router = Linear(place_projection(router, engine_dtype, device),
                             None if bias is None else place_vector(bias, device))
        if self.shared is not None and self.shared.in_dtype != self.router.in_dtype:
            raise ValueError("the shared expert and the router read their input in one dtype")
        self.correction = None if n["correction"] is None else place_vector(tensors[n["correction"]], device)
        sides = {side: [tensors[n["expert_" + side].format(e=e)] for e in range(self.experts)]
                 for side in (("gate", "up", "down") if self.gated else ("up", "down"))}
        limits = [limit] * self.experts
        if self.always:
            m, sfx = part_class("feed_forward", shared.kind)._names(shared), shared.get("weight_suffix", ".weight")
            for side in sides:
                sides[side].append(tensors[m[side] + sfx])
            limits.append(float(shared.get("limit", 0.0)))
        self.used, self.n_experts = self.top + self.always, self.experts + self.always      # a token's, and all of them
        self.limits = place_vector(torch.tensor(limits), device) if limit else None
        self.fused = False
        if not self.experts:
            self.up = self.down = None
            return
        wide = (engine_dtype == torch.float32 or self.width % 8 or self.router.in_dtype == torch.float32
                or any(t.dtype == torch.float32 for side in sides.values() for t in side))
        # Hidden units of zero weight (act(0) = 0 goes through zero columns of the way back) fill a hidden width up: the
        # bfloat16 products walk K in steps of 8, and gate and up go through one of them in blocks of 32 rows, whose
        # epilogue gates. In float32 a launch behind the product gates, the up rows following all gate rows.
        self.fused = self.gated and not wide
        step = 32 if self.fused else 1 if engine_dtype == torch.float32 else 8
        F = -(-max(t.shape[0] for t in sides["up"]) // step) * step
        pad = torch.nn.functional.pad
        stacked = {side: torch.stack([pad(t, (0, F - t.shape[1]) if side == "down" else (0, 0, 0, F - t.shape[0])) for t in ts])
                   for side, ts in sides.items()}
        if wide:            # (a tensor kept in float32, or a width that the bfloat16 products do not take)
            stacked = {side: t.to(torch.float32) for side, t in stacked.items()}
        up = stacked["up"]
        if self.fused:
            blocks = [stacked[side].view(self.n_experts, F // 32, 32, self.width) for side in ("gate", "up")]
            up = torch.stack(blocks, dim=2).reshape(self.n_experts, 2 * F, self.width)
        elif self.gated:
            up = torch.cat([stacked["gate"], up], dim=1)
        self.hidden_rows = F
        self.up = place_matrix(up, engine_dtype, device)
        self.down = place_matrix(stacked["down"], engine_dtype, device)
        # where an entry's row is its own number: the products of few tokens (as many entries as those take)
        self.own_slots = torch.arange(128, dtype=torch.int32, device=device)

    @classmethod
    def _joins_experts(cls, spec: PartSpec, shared: PartSpec) -> bool:
        """Whether the shared expert runs as one expert more in the experts' own products: it is added as it is, it has
        their activation, and filling all of them up to one hidden width costs at most a fifth in weights and work."""
        if (cls._names(spec)["shared_gate"] is not None or spec.get("identity", 0) or spec.get("weigh", "output") != "output"
                or shared.kind != spec.get("activation", "relu2") or shared.kind not in GATED
                or shared.get("alpha") != spec.get("alpha") or float(shared.get("out_scale", 1.0)) != 1.0):
            return False
        X, top, a, b = spec["experts"], spec["top"], spec["hidden"], shared["hidden"]
        F = max(a, b)
        return (X + 1) * F <= 1.2 * (X * a + b) and (top + 1) * F <= 1.2 * (top * a + b)

    @property
    def in_dtype(self) -> torch.dtype:
        return self.router.in_dtype

    @property
    def forward_rows(self):
        """Everything but the weighted sum over a token's experts: for a block whose next launch (a norm on
        this part's result) makes that sum itself. None where the result is more than that sum."""
        return None if self.shared is not None else self._rows

    @property
    def forward_parts(self):
        """As `forward_rows`, with the shared expert's result beside the rows, for a block whose next launch adds both.
        None where that result is multiplied by a gate first, or the experts' weights are spent on their input."""
        return None if self.weigh == "input" or (self.shared is not None and self.shared_gated) else self._parts

    def router_ride(self, ctx: StepContext, T: int) -> Optional[RouterRide]:
        """The router, for the norm that hands this part its rows; None where it goes a launch of its own. The products then go
        by the tokens' choices: the plan, which takes all tokens, would be a launch again."""
        if (self.shared is not None or self.group_count > 1 or not self.fused or self.weigh != "output"
                or not ops.moe_direct_takes(T, self.used, self.n_experts)
                or not ops.moe_direct_pays(T, self.used, self.n_experts, self.width, self.hidden_rows)):
            return None
        ws = ctx.workspace
        return RouterRide(self.router.weight, self.router.bias, self.correction, self.top, self.always, self.scoring, self.normalize,
                          self.route_scale, ws.get("moe_choice", (T, self.used), torch.int32), ws.get("moe_weight", (T, self.used), torch.float32))

    def _parts(self, ctx: StepContext, n: torch.Tensor, routed: Optional[RouterRide] = None) -> RowsToCombine:
        extra: list = []
        r = self._rows(ctx, n, extra if self.shared is not None else None, routed)
        r.extra = extra[0] if extra else None
        return r

    def _rows(self, ctx: StepContext, n: torch.Tensor, shared_out: Optional[list] = None,
              routed: Optional[RouterRide] = None) -> RowsToCombine:
        T, top, used, X = n.shape[0], self.top, self.used, self.n_experts
        ws = ctx.workspace
        rules = dict(scoring=self.scoring, n_router=self.n_router, groups=self.group_count, keep=self.group_keep,
                     normalize=self.normalize, scale=self.route_scale, always=self.always)
        if self.shared is not None:
            # first, while the scratch it shares with the experts' products is free
            stream, ctx.stream = ctx.stream, None          # (its result is weighed before it is added anywhere)
            try:
                shared_out.append(self.shared.forward(ctx, n))
            finally:
                ctx.stream = stream
        # a prompt's router takes choice and plan along, where nothing else reads its logits
        rides = (routed is None and X > 0 and n.dtype == torch.bfloat16
                 and self.router.weight.dtype == torch.bfloat16 and not (self.shared is not None and self.shared_gated)
                 and ops.moe_router_takes(T, self.n_router, X, top, self.group_count, self.always, self.width)
                 and ops.moe_router_pays(T, self.n_router, top, self.width))
        z = None if routed is not None or rides else self.router(ctx, n, torch.float32, "router_logits")
        if shared_out is not None:
            shared_out.append(z)
        choice = ws.get("moe_choice", (T, used), torch.int32)
        weight = ws.get("moe_weight", (T, used), torch.float32)
        entries = T * used
        if routed is not None:
            hidden = ws.get("moe_hidden", (entries, self.hidden_rows), self.down.dtype)
            y = ws.get("moe_y", (entries, self.width), torch.float32)
            ops.moe_gemm_direct(n, self.up, hidden, choice, own_rows=True, epilogue="gated", limits=self.limits, alpha=self.alpha)
            ops.moe_gemm_direct(hidden, self.down, y, choice)
            return RowsToCombine(y, n, choice, weight, self.own_slots[:entries], X, by_entry=True)
        slot_of_entry = ws.get("moe_slot_of_entry", (entries,), torch.int32)
        y = ws.get("moe_y", (entries, self.width), torch.float32)
        if X:
            rows = ops.moe_tile_rows(entries, X, self.up.dtype)
            tiles = ws.get("moe_tiles", (ops.moe_max_tiles(entries, X, rows), 3), torch.int32)
            entry_of_slot = ws.get("moe_entry_of_slot", (entries,), torch.int32)
            if rides:
                counts = ws.get("moe_counts", (ops.moe_router_blocks(T), X), torch.int32)
                ops.moe_router_plan(n, self.router.weight, self.router.bias, self.correction, choice, weight, counts, top, X, rows,
                                    slot_of_entry, entry_of_slot, tiles, scoring=self.scoring, normalize=self.normalize,
                                    scale=self.route_scale, always=self.always)
            elif T <= ops.moe_route_plan_tokens():      # a decode step: choice and plan in one launch
                ops.moe_route_plan(z, self.correction, choice, weight, top, X, rows, slot_of_entry, entry_of_slot, tiles,
                                   **rules)
            else:
                ops.moe_route(z, self.correction, choice, weight, top, **rules)
                ops.moe_plan(choice, X, rows, slot_of_entry, entry_of_slot, tiles)
            hidden = ws.get("moe_hidden", (entries, self.hidden_rows), self.down.dtype)
            on_input = weight.view(-1) if self.weigh == "input" else None
            if self.fused:
                ops.moe_gemm(n, self.up, hidden, tiles, rows, entry_of_slot, gather_div=used, epilogue="gated",
                             limits=self.limits, alpha=self.alpha, weight=on_input)
            elif self.gated:
                both = ws.get("moe_gate_up", (entries, self.up.shape[1]), torch.float32, alias="mixer_in")
                ops.moe_gemm(n, self.up, both, tiles, rows, entry_of_slot, gather_div=used)
                ops.moe_gated(both, on_input, entry_of_slot, hidden, choice, self.limits, self.alpha)
            else:
                ops.moe_gemm(n, self.up, hidden, tiles, rows, entry_of_slot, gather_div=used, epilogue=self.activation)
            ops.moe_gemm(hidden, self.down, y, tiles, rows)
        else:
            ops.moe_route(z, self.correction, choice, weight, top, **rules)
        return RowsToCombine(y, n, choice, None if self.weigh == "input" else weight, slot_of_entry, X)

    def forward(self, ctx: StepContext, n: torch.Tensor) -> torch.Tensor:
        extra: list = []
        r = self._rows(ctx, n, extra if self.shared is not None else None)
        out = ctx.workspace.get("ffn_out", (n.shape[0], self.width), torch.float32)
        ops.moe_combine(r.y, r.h, r.choice, r.weight, r.slot_of_entry, r.n_experts, out)
        if self.shared is not None and self.shared_gated:
            y, z = extra
            ops.gated_row_add(out, y, z, self.n_router)
        elif self.shared is not None:
            for part in (extra[0] if extra[0].dim() == 3 else [extra[0]]):
                ops.add_rows(out, part)
        return out


register_part("feed_forward", "routed_experts", RoutedExperts)
