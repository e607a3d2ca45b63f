"""A linear map as the parts hold it: the matrix ``[out, in]`` in the compute dtype, the bias in float32."""
from __future__ import annotations

from typing import Optional

import torch

from .base import BuildEnv, StepContext


class RowsAhead:
    """Rows that a norm has yet to make out of the float32 ``x``: what ``Norm.ahead_of`` gives to the one product that reads them, whose kernel
    normalises them on the way. ``x`` stays as it is until that product has been launched."""

    __slots__ = ("x", "norm", "shape")

    def __init__(self, x: torch.Tensor, norm):
        self.x, self.norm, self.shape = x, norm, x.shape


class Linear:
    def __init__(self, weight: torch.Tensor, bias: Optional[torch.Tensor], layout: str, env: BuildEnv):
        """``layout``: "in_out" (stored [in, out], as GPT-2 checkpoints do) or "out_in"."""
        if layout not in ("in_out", "out_in"):
            raise ValueError(f"unknown weight layout {layout!r}")
        w = weight.to(env.device)
        if layout == "in_out":
            w = w.t()
        self.weight = w.to(env.dtype).contiguous()  # [out, in]
        self.bias = None if bias is None else bias.to(env.device, torch.float32).contiguous()
        self.n_out, self.n_in = self.weight.shape

    def takes_norm(self, kernels, rows: int) -> bool:
        """Whether the product of so many rows has a kernel that normalises them on the way."""
        takes = getattr(kernels, "takes_norm" if self.weight.dtype == torch.bfloat16 else "takes_norm_float32", None)
        return takes is not None and self.weight.data_ptr() % 16 == 0 and takes(rows, self.n_out, self.n_in)

    def __call__(self, a: torch.Tensor, ctx: StepContext, *, activation: str = "none", residual: Optional[torch.Tensor] = None,
                 out: Optional[torch.Tensor] = None, out_dtype: Optional[torch.dtype] = None, final: bool = False,
                 may_leave: bool = False) -> torch.Tensor:
        """``final``: the caller does not touch ``residual`` again in its ``forward``. Where the block allows it
        (``ctx.may_defer``) the product may then leave the sum of its K ranges to the norm that follows. ``may_leave`` (a
        float32 ``out`` without a residual): the product may leave its K ranges in ``ctx.product_pending`` for the kernel that
        reads ``out`` next."""
        if type(a) is RowsAhead:
            n = a.norm
            if (residual is None and not may_leave and (ctx.dtype if out is None and out_dtype is None else out_dtype or out.dtype) == self.weight.dtype
                    and self.takes_norm(ctx.kernels, a.shape[0])):
                if out is None:
                    out = ctx.empty(a.shape[0], self.n_out, out_dtype)
                ctx.kernels.linear_normed(a.x, n.weight, n.bias, n.eps, n.rms, self.weight, self.bias, out, activation)
                return out
            a = n(a.x, ctx)  # a product that the kernel is not for
        if ctx.pending is not None or ctx.product_pending is not None:
            ctx.settle()  # the unfinished product's ranges live in the workspace that this one is about to use
        if out is None:
            out = residual if residual is not None else ctx.empty(a.shape[0], self.n_out, out_dtype)
        if may_leave and residual is None and activation == "none" and out.dtype == torch.float32:
            ctx.product_pending = ctx.kernels.linear(a, self.weight, self.bias, out, may_leave_pending=True)
        elif final and ctx.may_defer and residual is out:
            ctx.pending = ctx.kernels.linear(a, self.weight, self.bias, out, activation=activation, residual=residual, may_leave_pending=True)
        else:
            ctx.kernels.linear(a, self.weight, self.bias, out, activation=activation, residual=residual)
        return out
