"""nn.Linear on the gfx950 kernels: short products (``t2t_linear``) and the
split-K weight gradient (``t2t_wgrad``).

The layers' projections (tunalab FlexSelfAttention's qkv / out projections
and GLU's gate_up / down, called from model/modules/layer.py:33-35) are
bias-free nn.Linear maps over all T tokens.  Over a short sequence their
forward and input gradient run on the tiles of ``t2t_linear``; over a long
one they are library products (hipBLASLt / rocBLAS through torch).  The
weight gradient dW = dY^T X contracts K = T rows into a small output
(768 x 768 ... 4096 x 768 over 16384 tokens), which the library runs on 36-192
output tiles, a fraction of the 256 CUs.  ``t2t_wgrad`` splits K across
work-groups into fp32 partials and sums them in a fixed order.
"""
from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _lib

_OUT_F32 = {torch.bfloat16: False, torch.float32: True}


def wgrad_applies(dy: torch.Tensor, x: torch.Tensor, weight: torch.Tensor) -> bool:
    """bf16 rows on a ROCm device, M and N multiples of 128, K of 64."""
    M, N = weight.shape
    K = x.numel() // max(N, 1)
    return (x.is_cuda and x.dtype == torch.bfloat16 and dy.dtype == torch.bfloat16
            and weight.dtype in _OUT_F32 and M % 128 == 0 and N % 128 == 0
            and K > 0 and K % 64 == 0)


def wgrad(dy: torch.Tensor, x: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    """dY^T X of [K, M] and [K, N] bf16 rows -> [M, N] (out_dtype)."""
    return _lib.host().wgrad(dy, x, _OUT_F32[out_dtype])


# Products of up to this many multiply-adds run on t2t_linear; the line is
# where its kernel takes as long as the library call's host side (~23 us;
# 2048 x 4096 x 768 = 6.4e9: 21 us), beyond which the library's kernels are
# faster (4096 x 2304 x 768 = 7.2e9: 24 against 19.5 us).
# Where nothing waits for the host (a captured graph, a full queue) only the
# kernels count: the input gradient's is 0 to 55 % faster than the library's
# up to here, with few exceptions (6144 x 768 x 768 14.2 against 13.4 us, 2048
# x 3072 x 1024 28.7 / 24.5), the forward's 5 to 40 % faster up to about 2.5e9
# (512 x 4096 x 1024 11.8 / 9.7) and up to 23 % slower from 3e9 on (3072 x
# 2304 x 768 20.7 / 15.9, 2048 x 4096 x 768 19.1 / 17.4).  The line does not
# move with that: a replayed graph has the bits of the eager call.
SHORT_PRODUCT = 6.5e9


def short_product(x: torch.Tensor, w: torch.Tensor, transposed: bool) -> bool:
    """Whether x W^T (x W when ``transposed``) of bf16 rows is t2t_linear's:
    small, contiguous, rows that aligned 16-byte pieces cover, operands under 2 GiB (a
    product with very few features could reach that), and not a call that a
    tracer, a mode or a tensor subclass has to see as torch's own."""
    if not (x.is_cuda and _lib.replaces_torch(x, w)):
        return False
    n, k = (w.shape[1], w.shape[0]) if transposed else w.shape
    rows = x.numel() // max(k, 1)
    return (x.device == w.device and x.dtype == torch.bfloat16
            and w.dtype == torch.bfloat16 and k > 0 and x.shape[-1] == k and k % 8 == 0
            and w.shape[1] % 8 == 0 and 0 < rows * n * k <= SHORT_PRODUCT
            and (rows + 128) * k < 1 << 30 and (w.shape[0] + 128) * w.shape[1] < 1 << 30
            and x.is_contiguous() and w.is_contiguous()
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
            and not torch.is_autocast_enabled())


def product(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """F.linear(x, w) of tensors that autograd does not watch."""
    if short_product(x, w, False):
        return _lib.host().linear(x, w, False)
    return F.linear(x, w)


class WGradLinearFn(torch.autograd.Function):
    """y = x W^T (bias-free): y and dX = dY W on t2t_linear for short
    sequences, by the library for long ones; dW by t2t_wgrad."""

    @staticmethod
    def forward(ctx, x, weight):
        ctx.save_for_backward(x, weight)
        return product(x, weight)

    @staticmethod
    def backward(ctx, dy):
        x, weight = ctx.saved_tensors
        dx = dw = None
        if ctx.needs_input_grad[0]:
            if _lib.unwatched(dy, weight) and short_product(dy, weight, True):
                dx = _lib.host().linear(dy, weight, True)
            else:
                dx = (dy.reshape(-1, dy.shape[-1]) @ weight.to(dy.dtype)).view(x.shape)
        if ctx.needs_input_grad[1]:
            if wgrad_applies(dy, x, weight):
                dw = wgrad(dy, x, weight.dtype)
            else:
                d2, x2 = dy.reshape(-1, dy.shape[-1]), x.reshape(-1, x.shape[-1])
                dw = (d2.t() @ x2).to(weight.dtype)
        return dx, dw


class Linear(nn.Linear):
    """nn.Linear (same parameters and state dict); bias-free bf16 maps on the
    GPU run as WGradLinearFn does."""

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        # (graphs being compiled keep torch's own linear: the Function's
        # backward calls the library through its host module)
        if (self.bias is None and x.is_cuda and x.dtype == torch.bfloat16
                and self.weight.dtype == torch.bfloat16 and not torch.compiler.is_compiling()):
            if _lib.unwatched(x, self.weight):
                return product(x, self.weight)
            return WGradLinearFn.apply(x, self.weight)
        return super().forward(x)
