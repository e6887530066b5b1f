"""The C++ host side of the per-layer calls: what it refuses before it reaches
a kernel, and when it may be called at all.  No call gets as far as a launch."""
import os
import subprocess
import sys
import threading
import time

import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as fwad
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils._python_dispatch import TorchDispatchMode
from torch.utils.flop_counter import FlopCounterMode

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


class _Plain(torch.Tensor):
    """A subclass without any behaviour of its own."""


class _Through(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _Seen(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def _answers(x):
    return _lib.unwatched(x), _lib.host().plain(x)


def test_plain_calls_are_unwatched():
    x = torch.zeros(2, 8)
    w = torch.nn.Parameter(x.clone())
    assert _answers(x) == (True, True) and _answers(w) == (False, True)
    with torch.no_grad():
        assert _lib.unwatched(x, w, x.t(), x[1:]) and _lib.replaces_torch(x, w)
        with torch.device("cpu"):
            assert _lib.replaces_torch(x, w)
        with _Seen():
            assert not _lib.replaces_torch(x, w)
    with torch.inference_mode():
        assert _lib.unwatched(torch.zeros(2))


@torch.no_grad()
def test_tracers_modes_and_transforms_watch():
    x = torch.zeros(2, 8)
    got = {}

    def look(name):
        def f(t):
            got[name] = _answers(t)
            return t * 2
        return f

    torch.jit.trace(look("jit"), x, check_trace=False)
    make_fx(look("make_fx"))(x)
    make_fx(look("make_fx fake"), tracing_mode="fake")(x)
    torch.func.vmap(look("vmap"))(x)
    torch.func.functionalize(look("functionalize"))(x)
    with FakeTensorMode(allow_non_fake_inputs=True) as fake:
        look("fake mode")(x)
    look("fake tensor")(fake.from_tensor(x))
    for name, mode in (("flops", FlopCounterMode(display=False)), ("mode", _Through())):
        with mode:
            look(name)(x)
    look("subclass")(x.as_subclass(_Plain))
    look("lazily negated")(torch._neg_view(x))
    look("sparse")(x.to_sparse())
    look("sparse rows")(x.to_sparse_csr())
    look("nested")(torch.nested.nested_tensor([x[0], x[1, :3]]))
    assert len(got) == 14
    assert not {n: a for n, a in got.items() if a != (False, False)}
    with fwad.dual_level():
        assert not _lib.unwatched(x)


def test_batched_gradients_watch():
    """torch.autograd.grad(is_grads_batched=True) hands a backward batched
    tensors without a function transform around it."""
    seen = []

    class Double(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x * 2

        @staticmethod
        def backward(ctx, dy):
            seen.append(_answers(dy))
            return dy * 2

    x = torch.zeros(3, requires_grad=True)
    torch.autograd.grad(Double.apply(x), x, torch.eye(3), is_grads_batched=True)
    assert seen == [(False, False)]


def test_host_calls_release_the_gil():
    """Another Python thread runs while a call of the host module is under way
    (a launch that waits on a full queue would stop it otherwise).  The switch
    interval keeps the interpreter itself from handing the GIL over."""
    x, host = torch.zeros(4, 128, dtype=torch.bfloat16), _lib.host()
    go, ran = threading.Lock(), []
    go.acquire()

    def other():
        with go:
            ran.append(True)

    before = sys.getswitchinterval()
    thread = threading.Thread(target=other)
    thread.start()
    try:
        sys.setswitchinterval(1000.0)
        end = time.perf_counter() + 5.0
        go.release()
        while not ran and time.perf_counter() < end:
            try:
                host.swiglu(x)  # refused: host memory
            except RuntimeError:
                pass
        assert ran
    finally:
        sys.setswitchinterval(before)
        thread.join()


@pytest.mark.parametrize("heads", [0, -2])
def test_rope_refuses_a_head_count_that_is_not_positive(heads):
    """An integer division by zero would end the process."""
    code = ("import torch, tagseq2tagseq_amd.rope as r\n"
            "t = torch.zeros(8, 32)\n"
            "try:\n"
            f"    r.qkv_rope(torch.zeros(1, 8, 384, dtype=torch.bfloat16), t, t, {heads})\n"
            "except ValueError as e:\n"
            "    assert 'num_heads' in str(e), e\n"
            "    print('refused')\n")
    got = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True,
                         cwd=os.path.dirname(_lib.HERE))
    assert got.stdout == "refused\n", (got.returncode, got.stderr[-500:])


def test_overwriting_token_inputs_needs_the_words_too():
    lists = TokenLists(128, [[DocSpan(0, 0, 128)]], torch.device("cpu"), words=1,
                       link_rows=[np.ones((1, 1), dtype=np.uint64)])
    with pytest.raises(RuntimeError, match="q_bits and kv_bits are needed"):
        lists.build((torch.zeros(1, 128, dtype=torch.int32), None, None))


@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("shape", [(1, 2, 128, 64, 1), (2, 128, 64)])
def test_rope_backward_refuses_gradients_of_other_ranks(which, shape):
    t = [torch.zeros(1, 2, 128, 64, dtype=torch.bfloat16) for _ in range(3)]
    t[which] = torch.zeros(shape, dtype=torch.bfloat16)
    cs = torch.zeros(128, 32)
    with pytest.raises(ValueError, match="4-D"):
        _lib.host().qkv_rope_backward(*t, cs, cs, 0)
