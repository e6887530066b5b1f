"""SwiGLU of the layers' MLP on the gfx950 kernels (``t2t_swiglu`` and its
gradient): h = silu(g) * u from the gate / up product [g | u], one pass
forward, one pass backward writing the product's gradient [dg | du] whole.

Replaces the activation and product of tunalab's GLU(activation="silu") in
the reference's layers (model/modules/layer.py:23-28; textbook definition,
parity with tunalab unpinned), which torch runs as chunk + silu + multiply
and, backward, four elementwise kernels and a concatenation.
"""
from __future__ import annotations

import torch

from . import _lib


def swiglu_applies(gu: torch.Tensor) -> bool:
    """bf16 rows [..., 2H] on a ROCm device with H % 8 == 0."""
    return gu.is_cuda and gu.dtype == torch.bfloat16 and gu.shape[-1] % 16 == 0


class SwiGLUFn(torch.autograd.Function):
    """forward(gu [..., 2H]) -> silu(gu[..., :H]) * gu[..., H:] ([..., H])."""

    @staticmethod
    def forward(ctx, gu):
        h, rows = _lib.host().swiglu(gu)
        ctx.save_for_backward(rows)
        ctx.shape = gu.shape
        return h

    @staticmethod
    def backward(ctx, dh):
        (rows,) = ctx.saved_tensors
        return _lib.host().swiglu_backward(rows, dh, ctx.shape)


def swiglu_rows(gu: torch.Tensor) -> torch.Tensor:
    """SwiGLU of rows that swiglu_applies accepts."""
    if _lib.unwatched(gu):
        return _lib.host().swiglu(gu)[0]
    return SwiGLUFn.apply(gu)


def swiglu(gu: torch.Tensor) -> torch.Tensor:
    """silu(g) * u of [g | u] rows on the fused kernels (bf16, ROCm device)."""
    if not swiglu_applies(gu):
        raise RuntimeError("swiglu needs bf16 rows on a ROCm device with H % 8 == 0")
    return swiglu_rows(gu)
