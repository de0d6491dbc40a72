"""RMS norm: y = x * rsqrt(mean(x^2) + eps) * w, no offset, no bias
(/root/reference/crates/imparo-cpu/src/ops.rs:6-22). The residual add that
precedes a norm is fused into it (the reference's add_rms_norm,
/root/reference/crates/imparo-backend/src/lib.rs:2603-2609).

With `groups` > 1 the row is cut into that many equal consecutive parts and
each is divided by its own root mean square; the weight spans the whole row.
`tensor` names the weight outright where a checkpoint does not call it
`<prefix>.weight`. `offset` is added to the stored weight (1 where a file keeps a weight's
distance from one). `scale_tensor` names a second vector of the row's width and
`multiplier` a constant that the normed row is multiplied by as well (a layer
scale and a residual multiplier on a norm that sits behind a sublayer): all
three are folded into one float32 weight when the model is loaded. `scalar`: the
stored weight is a single number for the whole row (a tensor without
dimensions), spread over the row's width when the model is loaded.

A block may leave its sublayer's result pending on the stream together with
the norm it goes through before the add (`Residual.post`); this norm then
applies that norm, adds, and norms the sum in one launch."""
from __future__ import annotations

from typing import Dict, Optional

import torch

from ..config.plan import PartSpec
from ..kernels import ops
from ..weights.loader import TensorDecl
from .base import Declared, Residual, StepContext, one_delta
from .linear import place_vector
from .registry import register_part


class LinkedNorm:
    """What a norm over whole rows needs to read a stream kept as several copies of a row (hyper-connections): the
    class says its `row_norm()`, (kind, weight, bias, eps) as the stream kernel takes it."""
    routes = True         # `forward_linked` may take a mixture's router into its launch

    def row_norm(self):
        raise NotImplementedError

    def _read(self, ctx: StepContext, res: Residual, link, out: torch.Tensor, rows: Optional[torch.Tensor] = None, route=None):
        """norm(sum_t read[t] x'_t) with x' the copies behind the pending add, into `out`; without `rows` the copies
        are moved on. `link` None: the plain sum of the copies is read."""
        kind, weight, bias, eps = self.row_norm()
        x = res.x if res.streams is None else res.streams
        if res.pending is None:
            return ops.stream_norm(x, kind, weight, bias, eps, out, read=None if link is None else link.read, rows=rows,
                                   streams=link.streams if link is not None else None)
        if res.link is None or res.post is not None or isinstance(res.pending, tuple):
            raise ValueError("what joins several copies of a stream is one delta that goes through no norm of its own")
        n = res.link.streams
        if link is not None and link.streams != n:
            raise ValueError(f"a stream of {n} copies cannot be read as {link.streams}")
        moved = None
        if rows is None:
            moved = ctx.workspace.get("streams", (res.x.shape[0], n, res.x.shape[1]), torch.float32)
        if (route is not None and rows is None and out.dtype == torch.bfloat16
                and ops.stream_step_routes(x, res.pending, n, weight, bias, route.weight, route.top)):
            route.done = True
        ops.stream_norm(x, kind, weight, bias, eps, out, delta=res.pending, mix=res.link.mix, join=res.link.join,
                        read=None if link is None else link.read, x_out=moved, rows=rows,
                        route=route if route is not None and route.done else None)
        if rows is None:
            res.streams, res.pending, res.link = moved, None, None
        return out

    def forward_linked(self, ctx: StepContext, res: Residual, link, out_dtype: torch.dtype,
                       name: str = "normed", route=None) -> torch.Tensor:
        """`forward` for a sublayer with a link of its own: the normed sum of the copies, weighed by its `read`. `route`: the
        sublayer's router, which the launch takes along where it can."""
        more = {} if route is None else dict(route=route)        # (a norm with a `_read` of its own may know no routers)
        return self._read(ctx, res, link, ctx.workspace.get(name, tuple(res.x.shape), out_dtype), **more)


class RmsNorm(LinkedNorm):
    role = "norm"
    graph_safe = True     # launches kernels only: a step made of such parts can be captured

    @staticmethod
    def _tensor(spec: PartSpec) -> str:
        return spec.get("tensor") or f"{spec.prefix}.weight"

    @classmethod
    def declare(cls, spec: PartSpec) -> Declared:
        # a weight that an offset of 1 is added to is drawn near zero
        shape = () if spec.get("scalar") else (spec["width"],)
        out = {cls._tensor(spec): (TensorDecl(shape, "vector"), "bias" if spec.get("offset") else "norm")}
        if spec.get("scale_tensor"):
            out[spec["scale_tensor"]] = (TensorDecl((spec["width"],), "vector"), "norm")
        return out

    def __init__(self, spec: PartSpec, tensors: Dict[str, torch.Tensor], device: torch.device,
                 engine_dtype: torch.dtype):
        self.width = spec["width"]
        self.eps = float(spec["eps"])
        self.groups = int(spec.get("groups") or 1)
        if self.groups < 1 or self.width % self.groups:
            raise ValueError(f"a norm over {self.width} values cannot be cut into {self.groups} equal parts")
        weight = tensors[self._tensor(spec)].to(torch.float32) + float(spec.get("offset") or 0.0)
        if spec.get("scalar"):
            weight = weight.reshape(1).expand(self.width)
        if spec.get("scale_tensor"):
            weight = weight * tensors[spec["scale_tensor"]].to(torch.float32)
        if spec.get("multiplier") is not None:
            weight = weight * float(spec["multiplier"])
        self.weight = place_vector(weight, device)

    def row_norm(self):
        if self.groups != 1:
            raise ValueError("a norm that reads several copies of a stream does not cut rows into groups")
        return "rms", self.weight, None, self.eps

    def as_post(self):
        """(weight, eps) for `Residual.post`: this norm applied to a sublayer's result by whoever adds it."""
        if self.groups != 1:
            raise ValueError("a norm behind a sublayer does not cut rows into groups")
        return self.weight, self.eps

    def forward(self, ctx: StepContext, res: Residual, out_dtype: torch.dtype, name: str = "normed") -> torch.Tensor:
        """Adds the pending delta into the stream (if any) and returns the
        normed rows in `out_dtype`."""
        out = ctx.workspace.get(name, tuple(res.x.shape), out_dtype)
        one_delta(res)
        pending, res.pending = res.pending, None
        post, res.post = res.post, None
        if post is not None and pending is not None:
            if self.groups > 1:
                raise ValueError("a norm in groups cannot take a sublayer's result through a norm of its own")
            ops.post_norm_add(res.x, pending, post[0], post[1], self.weight, self.eps, out)
        elif self.groups > 1:
            ops.group_rms_norm(res.x, self.weight, self.groups, self.eps, out, delta=pending,
                               write_back=pending is not None)
        elif pending is not None:
            ops.rms_norm(res.x, self.weight, self.eps, out, delta=pending, write_back=True)
        else:
            ops.rms_norm(res.x, self.weight, self.eps, out)
        return out

    def forward_shifted(self, ctx: StepContext, res: Residual, out_dtype: torch.dtype, mix: torch.Tensor,
                        state: torch.Tensor, name: str = "normed") -> torch.Tensor:
        """`forward` for a step whose rows all bring one token, with the token shift behind the norm in
        the same launch: out = h + (prev - h) * mix, where the request's prev (state[slot]) becomes h."""
        out = ctx.workspace.get(name, tuple(res.x.shape), out_dtype)
        if res.post is not None:
            raise ValueError("the norm with the token shift does not take a sublayer's result through a norm of its own")
        one_delta(res)
        pending, res.pending = res.pending, None
        ops.group_rms_norm(res.x, self.weight, self.groups, self.eps, out, delta=pending,
                           write_back=pending is not None, shift_mix=mix, shift_state=state, slot=ctx.slot)
        return out

    def can_emit(self) -> bool:
        return self.groups == 1

    def emit(self, program, out_dtype: torch.dtype) -> None:
        """Appends `forward` to a native step program."""
        if self.groups != 1:
            raise ValueError("the step program's norm does not cut rows into groups")
        program.norm(self.weight, self.eps, self.width, out_dtype)

    def emit_head(self, program, head_linear) -> None:
        """Appends `forward_rows` followed by the head's projection."""
        program.head(self.weight, self.eps, self.width, head_linear)

    def forward_rows(self, ctx: StepContext, res: Residual, rows: torch.Tensor, out_dtype: torch.dtype,
                     name: str = "normed_rows") -> torch.Tensor:
        """Norm of selected rows only (the rows whose logits are wanted); the
        stream itself is left as it is."""
        out = ctx.workspace.get(name, (rows.shape[0], self.width), out_dtype)
        if res.link is not None or res.streams is not None:
            return self._read(ctx, res, None, out, rows)
        one_delta(res)
        if res.post is not None and res.pending is not None:
            if self.groups > 1:
                raise ValueError("a norm in groups cannot take a sublayer's result through a norm of its own")
            ops.post_norm_add(res.x, res.pending, res.post[0], res.post[1], self.weight, self.eps, out, rows=rows)
        elif self.groups > 1:
            ops.group_rms_norm(res.x, self.weight, self.groups, self.eps, out, delta=res.pending, rows=rows)
        else:
            ops.rms_norm(res.x, self.weight, self.eps, out, delta=res.pending, rows=rows)
        return out


class LayerNorm(LinkedNorm):
    """y = (x - mean) / sqrt(mean((x - mean)^2) + eps) * w + b over the row, in float32. What is pending on the stream is
    added in the same launch. Parameters: width, eps, tensor (the weight's name; the bias is `<tensor>.b`), multiplier
    (a constant that the result is multiplied by, folded into weight and bias)."""
    role = "norm"
    graph_safe = True     # launches kernels only: a step made of such parts can be captured

    @staticmethod
    def _tensors(spec: PartSpec):
        base = spec.get("tensor") or f"{spec.prefix}.weight"
        return base, f"{base}.b"

    @classmethod
    def declare(cls, spec: PartSpec) -> Declared:
        w, b = cls._tensors(spec)
        return {w: (TensorDecl((spec["width"],), "vector"), "norm"), b: (TensorDecl((spec["width"],), "vector"), "bias")}

    def __init__(self, spec: PartSpec, tensors: Dict[str, torch.Tensor], device: torch.device,
                 engine_dtype: torch.dtype):
        w, b = self._tensors(spec)
        self.width, self.eps = spec["width"], float(spec["eps"])
        m = spec.get("multiplier")
        m = 1.0 if m is None else float(m)
        self.weight = place_vector(tensors[w].to(torch.float32) * m, device)
        self.bias = place_vector(tensors[b].to(torch.float32) * m, device)

    def row_norm(self):
        return "layer", self.weight, self.bias, self.eps

    def forward(self, ctx: StepContext, res: Residual, out_dtype: torch.dtype, name: str = "normed") -> torch.Tensor:
        """Adds what is pending into the stream (if anything) and returns the normed rows in `out_dtype`."""
        out = ctx.workspace.get(name, tuple(res.x.shape), out_dtype)
        if res.post is not None:
            raise ValueError("this norm does not take a sublayer's result through a norm of its own")
        one_delta(res)
        pending, res.pending = res.pending, None
        return ops.stream_norm(res.x, *self.row_norm(), out, delta=pending, x_out=None if pending is None else res.x)

    def forward_rows(self, ctx: StepContext, res: Residual, rows: torch.Tensor, out_dtype: torch.dtype,
                     name: str = "normed_rows") -> torch.Tensor:
        """Norm of the chosen rows only; the stream itself is left as it is."""
        out = ctx.workspace.get(name, (rows.shape[0], self.width), out_dtype)
        if res.link is not None or res.streams is not None:
            return self._read(ctx, res, None, out, rows)
        if res.post is not None:
            raise ValueError("this norm does not take a sublayer's result through a norm of its own")
        one_delta(res)
        return ops.stream_norm(res.x, *self.row_norm(), out, delta=res.pending, rows=rows)


class DynamicTanh:
    """A norm without a statistic: y = tanh(alpha x) * w + b with one number alpha for the whole row, w and b over the
    row's width. What is pending on the stream, one delta or two, is added in the same launch. Parameters: width,
    tensor (the weight's name; the others are `<tensor>.alpha`, without dimensions, and `<tensor>.b`)."""
    role = "norm"
    graph_safe = True     # launches kernels only: a step made of such parts can be captured

    @staticmethod
    def _tensors(spec: PartSpec):
        base = spec.get("tensor") or f"{spec.prefix}.weight"
        return base, f"{base}.alpha", f"{base}.b"

    @classmethod
    def declare(cls, spec: PartSpec) -> Declared:
        w, alpha, b = cls._tensors(spec)
        return {w: (TensorDecl((spec["width"],), "vector"), "norm"), alpha: (TensorDecl((), "vector"), "norm"),
                b: (TensorDecl((spec["width"],), "vector"), "bias")}

    def __init__(self, spec: PartSpec, tensors: Dict[str, torch.Tensor], device: torch.device,
                 engine_dtype: torch.dtype):
        w, alpha, b = self._tensors(spec)
        self.width = spec["width"]
        self.weight, self.bias = place_vector(tensors[w], device), place_vector(tensors[b], device)
        self.alpha = float(tensors[alpha].to(torch.float32).reshape(()))

    @staticmethod
    def _deltas(res: Residual):
        if res.post is not None:
            raise ValueError("this norm does not take a sublayer's result through a norm of its own")
        if res.pending is None:
            return ()
        return res.pending if isinstance(res.pending, tuple) else (res.pending,)

    def forward(self, ctx: StepContext, res: Residual, out_dtype: torch.dtype, name: str = "normed") -> torch.Tensor:
        """Adds what is pending into the stream (if anything) and returns the rows behind the norm in `out_dtype`."""
        normed, res.normed = res.normed, None
        if normed is not None and normed.norm is self and normed.out_dtype == out_dtype and res.pending is None:
            return normed.rows
        out = ctx.workspace.get(name, tuple(res.x.shape), out_dtype)
        deltas, res.pending = self._deltas(res), None
        return ops.dynamic_tanh(res.x, self.alpha, self.weight, self.bias, out, deltas, write_back=bool(deltas))

    def ride(self, x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], into: torch.Tensor,
             rows: torch.Tensor) -> torch.Tensor:
        """into += x . weight^T (+ bias), and `rows` the new stream behind this norm, in one launch (a part that has this
        method may ride with the product before it)."""
        return ops.rows_gemm_tanh(x, weight, into, bias=bias, out=rows, alpha=self.alpha, norm_weight=self.weight,
                                  norm_bias=self.bias)

    def forward_rows(self, ctx: StepContext, res: Residual, rows: torch.Tensor, out_dtype: torch.dtype,
                     name: str = "normed_rows") -> torch.Tensor:
        """The chosen rows behind the norm; the stream itself is left as it is."""
        out = ctx.workspace.get(name, (rows.shape[0], self.width), out_dtype)
        return ops.dynamic_tanh(res.x, self.alpha, self.weight, self.bias, out, self._deltas(res), rows=rows)


class NoNorm:
    """No norm where a block has a place for one: the sublayer reads the stream itself. What is
    pending on the stream is added first, through the norm it carries if it carries one, in the
    same launch that hands the rows on in the dtype the reader asks for."""
    role = "norm"
    graph_safe = True     # launches kernels only: a step made of such parts can be captured

    @classmethod
    def declare(cls, spec: PartSpec) -> Declared:
        return {}

    def __init__(self, spec: PartSpec, tensors: Dict[str, torch.Tensor], device: torch.device,
                 engine_dtype: torch.dtype):
        self.width = spec["width"]

    @staticmethod
    def _add_plain(res: Residual, pending) -> None:
        """A delta that carries no norm: its slices are added to the stream in order."""
        if not isinstance(pending, torch.Tensor):
            raise ValueError("rows that a routed feed-forward left to be combined go through a norm behind it")
        for part in (pending if pending.dim() == res.x.dim() + 1 else [pending]):
            ops.add_rows(res.x, part)

    def forward(self, ctx: StepContext, res: Residual, out_dtype: torch.dtype, name: str = "normed") -> torch.Tensor:
        one_delta(res)
        pending, res.pending = res.pending, None
        post, res.post = res.post, None
        if pending is not None and post is None:
            self._add_plain(res, pending)
            pending = None
        if pending is None and out_dtype == torch.float32:
            return res.x          # readers do not write into what they read
        out = ctx.workspace.get(name, tuple(res.x.shape), out_dtype)
        if pending is None:
            return ops.cast_rows(res.x, out)
        ops.post_norm_add(res.x, pending, post[0], post[1], None, 0.0, out)
        return out

    def forward_rows(self, ctx: StepContext, res: Residual, rows: torch.Tensor, out_dtype: torch.dtype,
                     name: str = "normed_rows") -> torch.Tensor:
        """The chosen rows as they would be after the pending add; the stream itself is left as it is."""
        out = ctx.workspace.get(name, (rows.shape[0], self.width), out_dtype)
        one_delta(res)
        if res.pending is None:
            return ops.cast_rows(res.x, out, rows)
        if res.post is None:
            raise ValueError("rows are chosen from a stream whose pending delta goes through a norm, or has none pending")
        ops.post_norm_add(res.x, res.pending, res.post[0], res.post[1], None, 0.0, out, rows=rows)
        return out


register_part("norm", "rms_norm", RmsNorm)
register_part("norm", "layer_norm", LayerNorm)
register_part("norm", "dynamic_tanh", DynamicTanh)
register_part("norm", "none", NoNorm)
