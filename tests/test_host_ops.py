"""The C++ host side of the per-layer calls: what it refuses before it reaches
a kernel.  None of these calls gets as far as a launch."""
import pytest
import torch

from tagseq2tagseq_amd import _lib, attention, norm, rope  # noqa: F401  (registers the ops)
from tagseq2tagseq_amd.mask_creators import TokenLists
from tagseq2tagseq_amd.synth import DocSpan


def _tables():
    one = torch.ones(1, 1, 1, dtype=torch.int32)
    return [one] * 12 + [torch.zeros(1, 2, 128, 4, dtype=torch.int32)]


def _host_tensor_calls():
    def rows(*shape):
        return torch.zeros(*shape, dtype=torch.bfloat16)

    q, lse, x, w = rows(1, 2, 128, 64), torch.zeros(1, 2, 128), rows(4, 128), rows(128)
    cs, ops, host = torch.zeros(128, 32), torch.ops.t2t, _lib.host()
    doc, words = torch.zeros(1, 128, dtype=torch.int32), torch.zeros(1, 0, 128, dtype=torch.int64)
    return {
        "masked_attention": lambda: ops.masked_attention(q, q, q, _tables(), 0.1),
        "masked_attention_backward": lambda: ops.masked_attention_backward(
            q, q, q, q, q, lse, _tables(), 0.1),
        "rms_norm": lambda: ops.rms_norm(x, w, 1e-6),
        "rms_norm_backward": lambda: ops.rms_norm_backward(x, x, w, torch.ones(4)),
        "qkv_rope": lambda: ops.qkv_rope(rows(1, 128, 384), cs, cs, 2, 0),
        "qkv_rope_backward": lambda: ops.qkv_rope_backward(q, q, q, cs, cs, 0),
        "swiglu": lambda: host.swiglu(x),
        "swiglu_backward": lambda: host.swiglu_backward(x, rows(4, 64), [4, 128]),
        "linear": lambda: host.linear(x, rows(64, 128), False),
        "wgrad": lambda: host.wgrad(rows(64, 128), rows(64, 128), True),
        "mask_meta": lambda: host.mask_meta(doc, words, words, 0),
        "token_inputs": lambda: TokenLists(128, [[DocSpan(0, 0, 128)]],
                                           torch.device("cpu")).build(),
    }


@pytest.mark.parametrize("name", sorted(_host_tensor_calls()))
def test_host_memory_is_refused(name):
    """A kernel that is handed an address of host memory faults the GPU."""
    with pytest.raises(RuntimeError, match="ROCm GPU tensors"):
        _host_tensor_calls()[name]()


@pytest.mark.parametrize("dtypes,error,match", [
    ((torch.float16,) * 5, NotImplementedError, "dtype Half"),
    ((torch.uint8,) * 5, NotImplementedError, "dtype Byte"),
    ((torch.float64,) * 5, NotImplementedError, "dtype Double"),
    ((torch.bfloat16, torch.float32, torch.bfloat16, torch.bfloat16, torch.bfloat16), ValueError,
     "differ in dtype"),
    ((torch.float32, torch.float32, torch.bfloat16, torch.float32, torch.float32), ValueError,
     "differ in dtype"),
])
def test_attention_ops_refuse_other_dtypes(dtypes, error, match):
    """The custom ops, which no caller validates for: 16-bit floats of another
    format would be read as bfloat16, narrower types past their end."""
    q, k, v, out, dout = (torch.zeros(1, 2, 128, 64, dtype=t) for t in dtypes)
    with pytest.raises(error, match=match):
        torch.ops.t2t.masked_attention(q, k, v, _tables(), 0.1)
    with pytest.raises(error, match=match):
        torch.ops.t2t.masked_attention_backward(q, k, v, out, dout, torch.zeros(1, 2, 128),
                                                _tables(), 0.1)


@pytest.mark.parametrize("which", [3, 4])
def test_attention_backward_refuses_another_dtype_of_out_or_its_gradient(which):
    t = [torch.zeros(1, 2, 128, 64, dtype=torch.bfloat16) for _ in range(5)]
    t[which] = t[which].float()
    with pytest.raises(ValueError, match="differ in dtype"):
        torch.ops.t2t.masked_attention_backward(*t, torch.zeros(1, 2, 128), _tables(), 0.1)
