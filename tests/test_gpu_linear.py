"""t2t_linear (short projections and their input gradient) against the float32
product of the same bf16 operands: ends of tiles and stages, every tile shape
of the dispatch, operands inside larger buffers of NaN, outputs of any
alignment; and the routes of linear.Linear."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from tagseq2tagseq_amd import _lib
from tagseq2tagseq_amd.linear import SHORT_PRODUCT, Linear, short_product

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _in_nan(rows, cols, pad, g):
    """[rows, cols] N(0, 1) inside a buffer of NaN, row stride cols + pad."""
    buf = torch.full((rows + 2, cols + pad), float("nan"), device=DEV, dtype=torch.bfloat16)
    buf[:rows, :cols] = torch.randn(rows, cols, generator=g, device=DEV).to(torch.bfloat16)
    return buf[:rows, :cols]


@pytest.mark.parametrize("transposed", [0, 1])
@pytest.mark.parametrize("M,N,K", [
    (1, 8, 8), (63, 64, 64), (64, 72, 56), (65, 136, 72), (130, 100, 128), (129, 200, 136),
    (300, 2730, 520), (257, 64, 1032),  # 64 x 64 tiles
    (2048, 1024, 72), (1921, 1032, 200),  # 128 x 64
    (4096, 2048, 40), (3969, 2056, 192),  # 128 x 128
])
def test_linear_against_float32(M, N, K, transposed):
    if transposed and N % 8:
        N += 8 - N % 8
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = _in_nan(M, K, 8, g)
    w = _in_nan(K, N, 16, g) if transposed else _in_nan(N, K, 16, g)
    out = torch.full((M + 1, N + 3), 7.0, device=DEV, dtype=torch.bfloat16)
    rc = _lib.lib().t2t_linear(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), transposed,
                               out.data_ptr(), out.stride(0), M, N, K,
                               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    _lib.check(rc, "t2t_linear")
    ref = x.float() @ (w.float() if transposed else w.float().t())
    # one bf16 rounding of a float32 sum of K products of N(0, 1) numbers
    torch.testing.assert_close(out[:M, :N].float(), ref, rtol=2.0 ** -8, atol=1e-6 * K)
    assert (out[M] == 7).all() and (out[:, N:] == 7).all()


def test_linear_refuses_what_it_cannot_address():
    t = torch.zeros(64, 64, device=DEV, dtype=torch.bfloat16)
    call = _lib.lib().t2t_linear
    assert call(t.data_ptr(), 64, t.data_ptr(), 64, 0, t.data_ptr(), 64, 64, 64, 60, None) == -2
    assert call(t.data_ptr() + 2, 64, t.data_ptr(), 64, 0, t.data_ptr(), 64, 8, 8, 8, None) == -1
    assert call(t.data_ptr(), 12, t.data_ptr(), 64, 0, t.data_ptr(), 64, 8, 8, 8, None) == -1
    assert call(t.data_ptr(), 1 << 24, t.data_ptr(), 64, 0, t.data_ptr(), 64, 64, 8, 8, None) == -2


@pytest.mark.parametrize("rows,din,dout", [(40, 128, 136), (7, 1365, 512), (33, 512, 2730)])
def test_linear_module_routes(rows, din, dout):
    """Widths that t2t_linear takes in both, one or no direction, against
    torch's own linear; autocast keeps torch's dtype."""
    lin = Linear(din, dout, bias=False).to(DEV, torch.bfloat16)
    x = torch.randn(2, rows, din, device=DEV).to(torch.bfloat16).requires_grad_(True)
    y = lin(x)
    dy = torch.randn_like(y)
    y.backward(dy)
    xr = x.detach().float().requires_grad_(True)
    yr = F.linear(xr, lin.weight.detach().float())
    yr.backward(dy.float())
    torch.testing.assert_close(y.float(), yr, rtol=2.0 ** -8, atol=1e-5 * din ** 0.5)
    torch.testing.assert_close(x.grad.float(), xr.grad, rtol=2.0 ** -8, atol=1e-5 * dout ** 0.5)
    with torch.no_grad():
        assert torch.equal(lin(x), y)
        with torch.autocast("cuda", dtype=torch.float16):
            assert lin(x).dtype == torch.float16
    assert short_product(x, lin.weight, False) == (din % 8 == 0)
    assert short_product(dy, lin.weight, True) == (din % 8 == 0 and dout % 8 == 0)
    big = int(SHORT_PRODUCT) // (din * dout) + 1
    assert not short_product(x.detach()[:1, :1].expand(1, big, din), lin.weight, False)


def _off_by_one(*shape):
    """Contiguous N(0, 1) rows that start one element past a 16-byte boundary."""
    n = 1
    for d in shape:
        n *= d
    buf = torch.randn(n + 8, device=DEV).to(torch.bfloat16)
    t = buf[1:1 + n].view(*shape)
    assert t.is_contiguous() and t.data_ptr() % 16 == 2
    return t


@pytest.mark.parametrize("din,dout", [(136, 72), (64, 200)])
def test_linear_of_rows_off_a_16_byte_boundary(din, dout):
    """Input rows and an incoming gradient that the kernel cannot read in whole
    pieces: torch's products, as for any other such operand."""
    lin = Linear(din, dout, bias=False).to(DEV, torch.bfloat16)
    x, dy = _off_by_one(40, din), _off_by_one(40, dout)
    want = F.linear(x.float(), lin.weight.float())
    with torch.no_grad():
        torch.testing.assert_close(lin(x).float(), want, rtol=2.0 ** -8, atol=1e-4)
    x = x.requires_grad_(True)
    y = lin(x)
    torch.testing.assert_close(y.float(), want, rtol=2.0 ** -8, atol=1e-4)
    y.backward(dy)
    torch.testing.assert_close(x.grad.float(), dy.float() @ lin.weight.float(), rtol=2.0 ** -8,
                               atol=1e-4)
    torch.testing.assert_close(lin.weight.grad.float(), dy.float().t() @ x.detach().float(),
                               rtol=2.0 ** -8, atol=1e-4)
