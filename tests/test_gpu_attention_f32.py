"""Float32 attention at the sizes where its decomposition can go wrong:
sequence ends inside a 32-row block, a tile and a row's list of 64 tiles, waves
without a block, grouped heads that walk a long column again.  Against the
float64 oracle (short) or the chunked float32 torch reference (long), at the
float32 parity bound of 1e-4."""
import dataclasses

import numpy as np
import pytest
import torch
from torch.nn.attention.flex_attention import create_block_mask

from tagseq2tagseq_amd.attention import flex_attention
from tagseq2tagseq_amd.block_mask import from_torch_block_mask
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


def _compact(bm):
    """The same mask with bitmap slots for the partial tiles' columns only, the
    last row's first: kv_bits_off is negative where a row's partial tiles start
    late, and no row's column 0 need have a slot."""
    Bm, nt = bm.kv_bits_off.shape
    partial = (bm.tile_class == 1).cpu()
    old_off, old_slot = bm.kv_bits_off.cpu(), bm.q_bits_slot.cpu()
    num, q_idx = bm.q_num_blocks[:, 0].cpu(), bm.q_indices[:, 0].cpu()
    off, slot = torch.zeros_like(old_off), torch.zeros_like(old_slot)
    new, used = {}, []
    for b in range(Bm):
        for r in reversed(range(nt)):
            cols = partial[b, r].nonzero()[:, 0].tolist()
            off[b, r] = len(used) - cols[0] if cols else len(used)
            for c in range(cols[0], cols[-1] + 1) if cols else ():
                new[b, r, c] = len(used)
                used.append(int(old_off[b, r]) + c)
        for c in range(nt):
            for i in range(int(num[b, c])):
                slot[b, c, i] = new[b, int(q_idx[b, c, i]), c]
    dev = bm.tile_bits.device
    return dataclasses.replace(bm, kv_bits_off=off.to(dev), q_bits_slot=slot.to(dev),
                               tile_bits=bm.tile_bits[torch.tensor(used, device=dev)], _c=None)


def _all_bits(bm, q, k, v, do):
    for t in (q, k, v):
        t.requires_grad_(True).grad = None
    out, lse = flex_attention(q, k, v, block_mask=bm, enable_gqa=True, return_lse=True)
    out.backward(do)
    return out.detach(), lse, q.grad, k.grad, v.grad


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T,max_doc", [(700, 250), (1500, 1500)])
def test_f32_slots_of_partial_tiles_only(T, max_doc, D, gpu_device):
    """A pool that holds the slots the header asks for and no other: partial
    tile (r, c) at kv_bits_off[r] + c, nothing for a full tile."""
    rng = np.random.default_rng(T)
    rows = [random_row(T, rng, words=1, uncovered=True, max_doc=max_doc) for _ in range(2)]
    bm = _mask_from_rows(rows, gpu_device)
    small = _compact(bm)
    assert small.tile_bits.shape[0] < bm.tile_bits.shape[0]
    args = _inputs(2, 4, 2, T, D, T, gpu_device, torch.float32)
    for a, b in zip(_all_bits(bm, *args), _all_bits(small, *args)):
        assert torch.equal(a, b)


def test_f32_full_tiles_without_a_slot(gpu_device):
    """A mask of full tiles only, whose rows' kv_bits_off is the end of the pool."""
    T = 256
    every = create_block_mask(lambda b, h, q, k: q >= 0, None, None, T, T, device=gpu_device)
    bm = from_torch_block_mask(every)
    assert (bm.tile_class == 2).all()
    end = dataclasses.replace(bm, kv_bits_off=torch.ones_like(bm.kv_bits_off),
                              tile_bits=bm.tile_bits[:1].clone(), _c=None)
    args = _inputs(1, 2, 1, T, 64, 3, gpu_device, torch.float32)
    got = _all_bits(end, *args)
    for a, b in zip(_all_bits(bm, *args), got):
        assert torch.equal(a, b)
    q, k, v = (t.detach()[0].double() for t in args[:3])
    p = torch.softmax(q @ k.transpose(-1, -2) * 64 ** -0.5, -1)
    assert_close(got[0][0], (p @ v).float(), F32_TOL, F32_TOL, "out")
