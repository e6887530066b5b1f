"""Float32 attention at the sizes where its decomposition can go wrong:
sequence ends inside a 32-row block, a tile and a row's list of 64 tiles, waves
without a block, grouped heads that walk a long column again.  Against the
float64 oracle (short) or the chunked float32 torch reference (long), at the
float32 parity bound of 1e-4."""
import numpy as np
import pytest
import torch

from tagseq2tagseq_amd.attention import flex_attention
from tests.helpers import assert_close, random_row, to_dev_words, torch_ref_attention
from tests.test_gpu_attention import F32_TOL, _inputs, _mask_from_rows, _oracle_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T", [1, 31, 32, 33, 127, 129, 160, 289])
def test_f32_block_and_tile_ends(T, D, gpu_device):
    rng = np.random.default_rng(T + D)
    rows = [random_row(T, rng, words=1, uncovered=T > 100, max_doc=70) for _ in range(2)]
    _oracle_check(rows, 2, 3, 1, T, D, seed=T, device=gpu_device, dtype=torch.float32)


@pytest.mark.parametrize("D,T,max_doc", [(64, 8448, 8448), (128, 8330, 3000)])
def test_f32_rows_of_more_than_64_tiles(D, T, max_doc, gpu_device):
    rng = np.random.default_rng(D)
    row = random_row(T, rng, words=0, uncovered=False, max_doc=max_doc)
    if max_doc == T:
        row = (np.zeros(T, dtype=np.int32), None, None)  # causal: 66 tiles in the last row
    bm = _mask_from_rows([row], gpu_device)
    q, k, v, do = _inputs(1, 2, 1, T, D, D, gpu_device, torch.float32)
    for t in (q, k, v):
        t.requires_grad_(True)
    out, lse = flex_attention(q, k, v, block_mask=bm, enable_gqa=True, return_lse=True)
    out.backward(do)
    bits = [to_dev_words(w, gpu_device) if w is not None else None for w in row[1:]]
    with torch.no_grad():
        ref = torch_ref_attention(q, k, v, do, [(torch.from_numpy(row[0]).to(gpu_device), *bits)])
    for h in range(2):
        assert_close(out[0, h].detach(), ref["o"][(0, h)], F32_TOL, F32_TOL, f"out {h}")
        assert_close(lse[0, h].detach(), ref["lse"][(0, h)], F32_TOL, F32_TOL, f"lse {h}")
        assert_close(q.grad[0, h], ref["dq"][(0, h)], F32_TOL, F32_TOL, f"dq {h}")
    assert_close(k.grad[0, 0], ref["dk"][(0, 0)], F32_TOL, F32_TOL, "dk")
    assert_close(v.grad[0, 0], ref["dv"][(0, 0)], F32_TOL, F32_TOL, "dv")
