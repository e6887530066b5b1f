"""GPU parity of the split-K weight gradient (t2t_wgrad, linear.Linear)
against a float32 torch reference of dY^T X, and determinism."""
import ctypes

import pytest
import torch

from tagseq2tagseq_amd import _lib
from tagseq2tagseq_amd.linear import Linear, WGradLinearFn, wgrad

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


@pytest.mark.parametrize("K,M,N,pad_a,pad_b", [(64, 128, 128, 0, 0), (192, 256, 384, 8, 16),
                                               (16384, 768, 768, 0, 0), (2048, 2304, 768, 0, 8),
                                               (16384, 4096, 768, 0, 0), (4096, 768, 2048, 16, 0)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_wgrad_against_float32(K, M, N, pad_a, pad_b, out_dtype):
    g = torch.Generator().manual_seed(K + M + N)
    dy = torch.randn(K, M + pad_a, generator=g).to(torch.bfloat16).to(DEV)[:, :M]
    x = torch.randn(K, N + pad_b, generator=g).to(torch.bfloat16).to(DEV)[:, :N]
    got = wgrad(dy, x, out_dtype)
    ref = dy.float().t() @ x.float()
    tol = 1e-4 * K ** 0.5 if out_dtype == torch.float32 else 8e-3 * float(ref.abs().max())
    torch.testing.assert_close(got.float(), ref, rtol=1e-3 if out_dtype == torch.float32 else 8e-3,
                               atol=tol)
    assert torch.equal(wgrad(dy, x, out_dtype), got)  # fixed summation order


# One step, fewer steps than buffers, step counts that the splits share out
# unevenly, grids that 8 does not divide, a row stride past 32 bits over the
# rows of a step.  A sum of K products of N(0, 1) is about sqrt(K); K roundings
# of 6e-8 of that in random directions give 6e-8 K (K = 6464: 4e-4), the
# largest of an output some five times as much: 1e-4 sqrt(K) (8e-3) holds
# that and is far below one product lost (about 1).
@pytest.mark.parametrize("K,M,N,lda", [(64, 128, 128, 128), (128, 128, 256, 256),
                                       (64 * 101, 384, 128, 384), (64 * 37, 640, 896, 640),
                                       (192, 128, 128, (1 << 24) + 8)])
def test_wgrad_uneven_splits_and_wide_rows(K, M, N, lda):
    g = torch.Generator().manual_seed(K + M)
    dy = torch.empty(K, lda, dtype=torch.bfloat16, device=DEV)[:, lda - M:]
    dy.copy_(torch.randn(K, M, generator=g))
    x = torch.randn(K, N, generator=g).to(torch.bfloat16).to(DEV)
    got = wgrad(dy, x, torch.float32)
    ref = dy.double().t() @ x.double()
    torch.testing.assert_close(got.double(), ref, rtol=0, atol=1e-4 * K ** 0.5)


def test_linear_gradients_match_nn_linear():
    torch.manual_seed(0)
    lin = Linear(256, 384, bias=False).to(DEV).to(torch.bfloat16)
    ref = torch.nn.Linear(256, 384, bias=False).to(DEV)
    ref.weight.data.copy_(lin.weight.data.float())
    x = torch.randn(2, 64, 256, device=DEV).to(torch.bfloat16)
    dy = torch.randn(2, 64, 384, device=DEV).to(torch.bfloat16)
    xa = x.clone().requires_grad_()
    y = lin(xa)
    assert type(y.grad_fn).__name__ == "WGradLinearFnBackward"
    y.backward(dy)
    xr = x.float().requires_grad_()
    ref(xr).backward(dy.float())
    torch.testing.assert_close(y.float(), ref(xr).detach(), rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(xa.grad.float(), xr.grad, rtol=2e-2, atol=5e-2)
    torch.testing.assert_close(lin.weight.grad.float(), ref.weight.grad, rtol=2e-2, atol=5e-2)


def test_rows_not_multiple_of_64_use_the_library_product():
    lin = Linear(128, 128, bias=False).to(DEV).to(torch.bfloat16)
    x = torch.randn(33, 128, device=DEV).to(torch.bfloat16).requires_grad_()
    lin(x).float().sum().backward()
    ref = torch.ones(33, 128, device=DEV).t() @ x.detach().float()
    torch.testing.assert_close(lin.weight.grad.float(), ref, rtol=2e-2, atol=5e-2)
