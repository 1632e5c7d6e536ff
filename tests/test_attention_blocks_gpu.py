"""Attention over blocks of sequences of any lengths in one launch, and the gather of a cached
context's keys and values."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from kgs.ops import decode as D
from kgs.ops import transformer as T

DEV = "cuda"


def test_block_items_order_and_refusals():
    it = T.block_items([(0, 256, 0, 0, 0), (256, 128, 0, 192, 1)], 384)
    assert it.tolist() == [[256, 0, 192, 1], [128, 0, 128, 0], [0, 0, 0, 0]]
    assert it.dtype == np.int32
    for bad in ((0, 100, 0, 0, 0), (0, 128, 0, 32, 1), (300, 128, 300, 0, 0), (0, 128, 0, 320, 0), (0, 0, 0, 0, 0)):
        with pytest.raises(ValueError):
            T.block_items([bad], 384)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv", [(8, 2), (3, 1), (4, 4)])
def test_blocks_match_per_sequence_bits(heads, kv):
    """The same tiles in the same order as one launch per sequence: equal bits. Prompts of one and
    several blocks beside chunks whose keys are in other buffers, at contexts that end on a
    block's edge and in its middle."""
    torch.manual_seed(heads)
    lens, past = [128, 384, 256], [(128, 64), (256, 320), (128, 1024)]
    rows = sum(lens) + sum(n for n, _ in past) + 5
    w = 128 * (heads + 2 * kv)
    qkv = torch.randn(rows, w, device=DEV).bfloat16()
    k = qkv[:, 128 * heads:128 * (heads + kv)]
    v = qkv[:, 128 * (heads + kv):]
    nk = sum(c + n for n, c in past)
    k2, v2 = torch.randn(2, nk, 128 * kv, device=DEV).bfloat16()
    seqs, want, r, kr = [], torch.zeros(rows, 128 * heads, device=DEV, dtype=torch.bfloat16), 0, 0
    for n in lens:
        seqs.append((r, n, r, 0, 0))
        T.attention_qkv(qkv[r:r + n], 1, n, heads, kv, out=want[r:r + n])
        r += n
    for n, c in past:
        seqs.append((r, n, kr, c, 1))
        want[r:r + n] = T.attention_chunk(qkv[r:r + n], k2[kr:kr + c + n], v2[kr:kr + c + n], heads, kv)
        r, kr = r + n, kr + c + n
    items = torch.from_numpy(T.block_items(seqs, rows)).to(DEV)
    out = torch.zeros_like(want)
    T.attention_blocks(qkv, k, v, items, heads, kv, out, k2, v2)
    assert torch.equal(out, want)
    assert not out[r:].any()  # rows of no item stay as they were


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("kv,ctx,rows", [(1, 1, 1), (2, 31, 64), (8, 32, 32), (8, 33, 160), (3, 500, 640), (2, 0, 33)])
def test_gather_kv_bits(fp8, kv, ctx, rows):
    """A copy: the bits of the tensor form, rows past the context zero, for whole and partial pages."""
    torch.manual_seed(ctx)
    cache = torch.randn(24, kv, 2, 4096, device=DEV)
    cache = cache.to(D.FP8) if fp8 else cache.bfloat16()
    pages = torch.randperm(24, device=DEV, dtype=torch.int32)[:18]
    k, v = torch.full((2, rows, 128 * kv), 7.0, device=DEV, dtype=torch.bfloat16)
    D.gather_kv_into(cache, pages, ctx, k, v)
    wk, wv = D.gather_kv(cache, pages, ctx, rows=rows)
    assert torch.equal(k, wk) and torch.equal(v, wv)
    with pytest.raises(ValueError):
        D.gather_kv_into(cache, pages[:0], 1, k, v)
