"""A dense projection y = x . W^T (+ b) on the GEMM kernels.

Not a part of its own: mixers, feed-forwards and the head are made of these.
The weight decides the kernel: a bfloat16 weight runs the MFMA kernels, a
float32 weight the float32 kernel; the input must already be in that dtype
(`in_dtype`), which the producer of the input asks for.
"""
from __future__ import annotations

from typing import Optional

import torch

from ..kernels import ops
from .base import StepContext

# Most of K where a product of at most 16 rows that sums the whole of K in a block and takes a norm without a statistic along beats
# slices of K and a launch for the norm, by how many blocks of eight weight rows the fullest CU has (one up to 2,048 weight rows, where
# up to 1,024 a block has four; every block reads all activations, so that the price goes by the blocks and by K). By the weight and K
# alone: a row's sums then come in one order in all steps of 1 to 16 rows. Measured in a graph, cold weights, us for 1 / 4 / 8 / 16 rows
# with the norm's launch counted in, riding and not: 1,024 weight rows over 1,024 3.7 3.9 4.0 4.3 and 5.6 5.8 5.9 6.0, over 3,072 5.4 5.8 6.2
# 7.1 and 6.4 6.6 6.7 6.9, over 3,584 16 rows 7.6 and 7.2; 2,048 over 4,096 7.5 7.7 8.2 9.4 and 8.6 8.8 9.1 9.4; 3,072 over 2,048 7.0 7.4 8.1 9.2
# and 8.5 8.6 8.8 9.3, over 3,072 16 rows 12.9 and 11.2; 5,120 over 1,024 6.1 6.4 6.9 8.1 and 7.8 8.1 8.1 8.5, over 2,048 16 rows 12.8 and
# 11.1; 8,192 over 512 6.9 and 7.5, over 1,024 10.3 and 9.0; 16,384 over 512 11.7 and 9.3.
RIDE_MAX_K = 4096
_RIDE_MOST_K = (4096, 2048, 1024, 512)


def _rides(weight_rows: int, k: int) -> bool:
    a_cu = -(-weight_rows // 2048)
    if a_cu > len(_RIDE_MOST_K):
        return False
    return k <= min(RIDE_MAX_K, 3072 if weight_rows <= 1024 else _RIDE_MOST_K[a_cu - 1])


class Linear:
    def __init__(self, weight: torch.Tensor, bias: Optional[torch.Tensor] = None):
        if weight.dim() != 2:
            raise ValueError(f"a projection weight is [out, in], got shape {list(weight.shape)}")
        self.weight = weight.contiguous()
        self.bias = None if bias is None else bias.to(torch.float32).contiguous()
        self.out_features, self.in_features = weight.shape

    @property
    def in_dtype(self) -> torch.dtype:
        return self.weight.dtype

    def __call__(self, ctx: StepContext, x: torch.Tensor, out_dtype: torch.dtype, name: str,
                 swiglu: bool = False, sliced_ok: bool = False, alias: Optional[str] = None,
                 into: Optional[torch.Tensor] = None, swiglu_scale: float = 1.0, limit: float = 0.0,
                 alpha: float = 1.0) -> torch.Tensor:
        """`swiglu`: the weight's rows alternate gate and up; the output is
        silu(gate) * up, half as wide (times `swiglu_scale`, before it is rounded), or with `limit` the
        unit with bounds that `ops.gemm` describes. `sliced_ok`: the caller's consumer adds
        slices, so the result may come as [slices, rows, out] sums over parts
        of K (few rows and a long K keep more of the chip busy that way).
        `alias`: the workspace group the output may share memory with.
        `into`: a float32 [rows, out] tensor the result may be added to instead
        (the residual stream); where the kernels do that, `into` itself is returned."""
        width = self.out_features // 2 if swiglu else self.out_features
        m = x.shape[0]
        ride = ctx.ride if into is not None else None
        if (ride is not None and not swiglu and m <= ops.ROWS_MAX and _rides(self.out_features, self.in_features) and x.dtype == torch.bfloat16
                and self.weight.dtype == torch.bfloat16 and self.in_features % 8 == 0 and ride.out_dtype == torch.bfloat16
                and into.dtype == torch.float32 and tuple(into.shape) == (m, width) and into.is_contiguous()):
            # a few rows: the product adds to the stream and takes the norm behind it along
            if ride.norm is None:
                return ops.rows_gemm_tanh(x, self.weight, into, bias=self.bias)
            ride.rows = ctx.workspace.get("normed", (m, width), ride.out_dtype)
            return ride.norm.ride(x, self.weight, self.bias, into, ride.rows)
        if sliced_ok and not swiglu and out_dtype == torch.float32:
            slices = ops.gemm_slices(m, self.out_features, self.in_features, self.weight.dtype)
            if slices > 1:
                out = ctx.workspace.get(name + "_sliced", (slices, m, width), out_dtype)
                return ops.gemm(x, self.weight, out, bias=self.bias)
        if (into is not None and not swiglu and out_dtype == torch.float32 and into.dtype == torch.float32
                and tuple(into.shape) == (m, width) and into.is_contiguous()
                and ops.gemm_adds(m, self.out_features, self.in_features, self.weight.dtype)):
            # one pass less over the rows for the norm that follows: the product's epilogue reads and writes the stream
            return ops.gemm(x, self.weight, into, bias=self.bias, add=True)
        out = ctx.workspace.get(name, (m, width), out_dtype, alias=alias)
        return ops.gemm(x, self.weight, out, bias=self.bias, swiglu=swiglu, swiglu_scale=swiglu_scale,
                        limit=limit, alpha=alpha)


def place_matrix(t: torch.Tensor, engine_dtype: torch.dtype, device: torch.device) -> torch.Tensor:
    """A matrix as the engine keeps it on the device: bfloat16 stays bfloat16
    under a bfloat16 engine, everything is float32 under a float32 engine, and
    a tensor stored in float32 stays float32 either way."""
    if engine_dtype == torch.float32 or t.dtype == torch.float32:
        return t.to(device=device, dtype=torch.float32).contiguous()
    return t.to(device=device, dtype=torch.bfloat16).contiguous()


def place_projection(t: torch.Tensor, engine_dtype: torch.dtype, device: torch.device) -> torch.Tensor:
    """`place_matrix` for a projection weight [out, in] whose inner size any model may choose: the
    bfloat16 kernels walk the inner size in steps of 8, so a weight over another inner size is kept in
    float32 and its projection runs the float32 kernel (whoever makes its input is asked for float32
    through `in_dtype`)."""
    if engine_dtype != torch.float32 and t.dim() == 2 and t.shape[1] % 8:
        t = t.to(torch.float32)
    return place_matrix(t, engine_dtype, device)


def place_vector(t: torch.Tensor, device: torch.device) -> torch.Tensor:
    """Norm weights, conv taps and biases are read as float32 by the kernels;
    widening bfloat16 to float32 is exact."""
    return t.to(device=device, dtype=torch.float32).contiguous()
