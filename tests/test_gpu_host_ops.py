"""The calls that go to the kernels without an autograd.Function (nothing to
record) against the same calls with one: equal bits, and still refused where
the Function refuses (forward-mode and function transforms) and still seen by
tracers, modes and subclasses; row strides and sizes that the C++ wrappers copy
or pass on."""
import math

import pytest
import torch
import torch.autograd.forward_ad as fwad
from torch._subclasses.fake_tensor import FakeTensor, FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils.flop_counter import FlopCounterMode

from tagseq2tagseq_amd import _lib, synth
from tagseq2tagseq_amd.attention import flex_attention
from tagseq2tagseq_amd.glu import swiglu
from tagseq2tagseq_amd.linear import Linear, short_product
from tagseq2tagseq_amd.mask_creators import create_doc_causal_block_mask
from tagseq2tagseq_amd.norm import rms_norm
from tagseq2tagseq_amd.rope import qkv_rope, rope_tables

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
T, H, D = 160, 2, 64


def _calls():
    g = torch.Generator(device=DEV).manual_seed(0)

    def rnd(*shape):
        return torch.randn(*shape, generator=g, device=DEV).to(torch.bfloat16)

    w = rnd(128)
    cos, sin = rope_tables(D, T, DEV)
    tokens = torch.zeros((1, T), dtype=torch.int64, device=DEV)
    mask = create_doc_causal_block_mask(tokens, synth.lognormal_docs(T, 50.0, 1.0, 90, 1).spans)
    k, v = rnd(1, H, T, D), rnd(1, H, T, D)
    lin = Linear(128, 256, bias=False).to(DEV, torch.bfloat16)
    return {
        "norm": (rnd(1, T, 128), lambda x: rms_norm(x, w, 1e-6)),
        "norm rows of a wider tensor": (rnd(1, T, 256)[..., :128], lambda x: rms_norm(x, w, 1e-6)),
        "rope": (rnd(1, T, 3 * H * D), lambda x: torch.cat(qkv_rope(x, cos, sin, H))),
        "swiglu": (rnd(1, T, 128), swiglu),
        "swiglu of transposed rows": (rnd(128, T).t(), swiglu),
        "attention": (rnd(1, H, T, D), lambda x: flex_attention(x, k, v, block_mask=mask)),
        "attention of [B, T, H, D] storage": (rnd(1, T, H, D).transpose(1, 2),
                                              lambda x: flex_attention(x, k, v, block_mask=mask)),
        "linear": (rnd(1, T, 128), lambda x: lin(x)),
    }


@pytest.mark.parametrize("name", [
    "norm", "norm rows of a wider tensor", "rope", "swiglu", "swiglu of transposed rows",
    "attention", "attention of [B, T, H, D] storage", "linear"])
def test_unrecorded_calls(name):
    x, call = _calls()[name]
    with torch.no_grad():
        plain = call(x)
        assert _lib.unwatched(x)
    recorded = call(x.detach().requires_grad_(True))
    assert plain.grad_fn is None and recorded.grad_fn is not None
    assert torch.equal(plain, recorded)
    with torch.no_grad(), fwad.dual_level():
        dual = fwad.make_dual(x, torch.ones_like(x))
        with pytest.raises((RuntimeError, NotImplementedError)):
            call(dual)
    with torch.no_grad(), pytest.raises(RuntimeError):
        torch.func.vmap(call)(torch.stack([x, x]))


@pytest.mark.parametrize("name", [
    "norm", "norm rows of a wider tensor", "rope", "swiglu", "swiglu of transposed rows",
    "attention", "attention of [B, T, H, D] storage"])
def test_traced_calls_run_again(name):
    """A trace holds the call itself, not the memory that its kernel filled."""
    x, call = _calls()[name]
    other = torch.randn_like(x)
    with torch.no_grad():
        traced = torch.jit.trace(call, x, check_trace=False)
        assert torch.equal(traced(other), call(other))
        assert torch.equal(traced(x), call(x))


def _short_linear():
    lin = Linear(128, 256, bias=False).to(DEV, torch.bfloat16)
    x = torch.randn(160, 128, device=DEV).to(torch.bfloat16)
    assert short_product(x, lin.weight, False)
    return lin, x


def test_linear_is_seen_by_tracers_modes_and_subclasses():
    lin, x = _short_linear()
    other = torch.randn_like(x)
    with torch.no_grad():
        want = torch.nn.functional.linear(other, lin.weight)
        assert torch.equal(torch.jit.trace(lin, x, check_trace=False)(other), want)
        graph = make_fx(lin)(x)
        assert torch.equal(graph(other), want)
        with FlopCounterMode(display=False) as flops:
            lin(x)
        assert flops.get_total_flops() == 2 * 160 * 128 * 256
        with FakeTensorMode(allow_non_fake_inputs=True) as fake:
            y = lin(fake.from_tensor(x))
        assert isinstance(y, FakeTensor) and y.shape == (160, 256)

        class Tagged(torch.Tensor):
            pass

        assert type(lin(x.as_subclass(Tagged))) is Tagged

        calls = []

        class Seen(torch.overrides.TorchFunctionMode):
            def __torch_function__(self, func, types, args=(), kwargs=None):
                calls.append(func)
                return func(*args, **(kwargs or {}))

        with Seen():
            assert torch.equal(lin(other), want)
        assert torch.nn.functional.linear in calls


def test_linear_batched_input_gradients():
    """Batched gradients of a frozen weight's map, as a Jacobian takes them."""
    lin, x = _short_linear()
    lin.weight.requires_grad_(False)
    x = x[:2].requires_grad_(True)
    dy = torch.randn(3, 2, 256, device=DEV).to(torch.bfloat16)
    got, = torch.autograd.grad(lin(x), x, dy, is_grads_batched=True)
    want = dy.float() @ lin.weight.float()
    torch.testing.assert_close(got.float(), want, rtol=2.0 ** -8, atol=1e-4)


def _off_by_one(*shape):
    """Contiguous N(0, 1) rows that start one element past a 16-byte boundary."""
    buf = torch.randn(math.prod(shape) + 8, device=DEV).to(torch.bfloat16)
    t = buf[1:1 + math.prod(shape)].view(*shape)
    assert t.is_contiguous() and t.data_ptr() % 16 == 2
    return t


def test_rows_off_a_16_byte_boundary_are_copied():
    """The kernels read rows in 16-byte pieces, and contiguous() of rows that
    are contiguous already is no copy."""
    x, dy = _off_by_one(3, 64, 256), _off_by_one(3, 64, 128)
    even = x.clone().requires_grad_(True)
    odd = x.requires_grad_(True)
    want, got = swiglu(even), swiglu(odd)
    assert torch.equal(want, got)
    want.backward(dy.clone())
    got.backward(dy)
    assert torch.equal(even.grad, odd.grad)
    x, host = x.detach(), _lib.host()
    norm_w = torch.randn(256, device=DEV).to(torch.bfloat16)
    assert torch.equal(rms_norm(x, norm_w, 1e-6), rms_norm(x.clone(), norm_w, 1e-6))
    assert torch.equal(host.wgrad(dy, x, True), host.wgrad(dy.clone(), x.clone(), True))
    w = _off_by_one(128, 256)
    assert torch.equal(host.linear(x, w, False), host.linear(x.clone(), w.clone(), False))
    assert torch.equal(host.linear(dy, w, True), host.linear(dy.clone(), w.clone(), True))


def test_linear_trains_on_rows_off_a_16_byte_boundary():
    """Widths whose weight gradient is the split kernel's."""
    lin = Linear(256, 128, bias=False).to(DEV, torch.bfloat16)
    x, dy = _off_by_one(128, 256), _off_by_one(128, 128)
    lin(x.requires_grad_(True)).backward(dy)
    torch.testing.assert_close(lin.weight.grad.float(), dy.float().t() @ x.detach().float(),
                               rtol=2.0 ** -8, atol=1e-3)


def test_library_errors_carry_their_message():
    with pytest.raises(RuntimeError, match="t2t_wgrad failed"):
        _lib.host().wgrad(torch.zeros(64, 100, device=DEV, dtype=torch.bfloat16),
                          torch.zeros(64, 128, device=DEV, dtype=torch.bfloat16), True)
