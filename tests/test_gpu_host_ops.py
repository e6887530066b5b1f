"""The calls that go to the kernels without an autograd.Function (nothing to
record) against the same calls with one: equal bits, and still refused where
the Function refuses (forward-mode and function transforms); row strides and
sizes that the C++ wrappers copy or pass on."""
import pytest
import torch
import torch.autograd.forward_ad as fwad

from tagseq2tagseq_amd import _lib, synth
from tagseq2tagseq_amd.attention import flex_attention
from tagseq2tagseq_amd.glu import swiglu
from tagseq2tagseq_amd.linear import Linear
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
    if name == "linear":
        return  # torch's own product differentiates either way
    with torch.no_grad(), fwad.dual_level():
        dual = fwad.make_dual(x, torch.ones_like(x))
        with pytest.raises((RuntimeError, NotImplementedError)):
            call(dual)
    with torch.no_grad(), pytest.raises(RuntimeError):
        torch.func.vmap(call)(torch.stack([x, x]))


def test_library_errors_carry_their_message():
    with pytest.raises(RuntimeError, match="t2t_wgrad failed"):
        _lib.host().wgrad(torch.zeros(64, 100, device=DEV, dtype=torch.bfloat16),
                          torch.zeros(64, 128, device=DEV, dtype=torch.bfloat16), True)
