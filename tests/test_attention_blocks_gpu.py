"""Attention over blocks of sequences of any lengths in one launch, and the gather of a cached
context's keys and values."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from kgs.models.llama import LlamaConfig
from kgs.ops import decode as D
from kgs.ops import transformer as T

DEV = "cuda"


def test_block_items_order_and_refusals():
    it = T.block_items([(0, 256, 0, 0, 0), (256, 100, 0, 190, 1)], 356)
    assert it.tolist() == [[256, 0, 190, 201], [128, 0, 128, 256], [0, 0, 0, 256]]
    assert it.dtype == np.int32
    for bad in ((300, 128, 300, 0, 0), (0, 128, 0, 320, 0), (0, 0, 0, 0, 0), (-1, 4, 0, 0, 0)):
        with pytest.raises(ValueError):
            T.block_items([bad], 384)


def test_prompt_rows_cpu():
    """What is dropped, where each row goes and which are wanted, for prompt portions and decode rows."""
    from kgs.serve.model import ServingModel

    class M:
        backend = "kgs"
        cfg = type("Cfg", (), {"heads": 8})

    seqs, dev = [(0, 20, 128, 0), (128, 130, 256, 64)], torch.device("cpu")
    p = ServingModel._prompt_rows(M, seqs, 387, dev, tail=3, wanted=[False, True])
    assert p.n == 153 and p.past == [(0, 194, 194, 1)]
    assert p.keep.tolist() == [*range(20), *range(128, 258), *range(384, 387)]
    assert p.last.tolist() == [149, 150, 151, 152]
    assert all(int(p.rows[k]) == i for i, k in enumerate(p.keep.tolist())) and int((p.rows >= 0).sum()) == 153
    assert sorted(map(tuple, p.items.tolist())) == [(0, 0, 0, 40), (20, 0, 64, 257), (148, 0, 192, 5)]
    for kw in ({"drop": False}, {}):  # kept whole where asked, or where no tile of rows is saved
        q = ServingModel._prompt_rows(M, seqs if kw else [(0, 120, 128, 0), (128, 128, 128, 0)], 384 if kw else 256, dev, **kw)
        assert q.keep is None and q.rows is None and q.last.tolist() == ([19, 257] if kw else [119, 255])
    assert q.items is None and q.n == 256  # equal portions: the batched launch


def test_split_items():
    """Every key tile of a block is in exactly one part, slots follow one another, short blocks and launches
    of many rounds stay whole."""
    it = T.block_items([(0, 300, 0, 3072, 1), (300, 256, 300, 0, 0)], 556)
    out, merges, slots = T.split_items(it, 32)
    got = {}
    for r, k0, pos, w in out.tolist():
        rows, part, parts, slot, t = w >> 1 & 255, w >> 9 & 15, w >> 13 & 15, w >> 17, (pos + (w >> 1 & 255) - 1) // 64 + 1
        got.setdefault((r, rows, pos, w & 1), []).append((t * part // parts, t * (part + 1) // parts, slot) if parts else (0, t, None))
    assert {k for k in got} == {(r, w >> 1, p, w & 1) for r, _, p, w in it.tolist()}
    for (r, rows, pos, _), ps in got.items():
        ps.sort()
        assert ps[0][0] == 0 and ps[-1][1] == (pos + rows - 1) // 64 + 1 and all(a[1] == b[0] for a, b in zip(ps, ps[1:]))
        assert (len(ps) > 1) == (pos >= 3072) and len({p[2] for p in ps}) == 1
    assert sorted(m[2] for m in merges.tolist()) == [sum(m[3] for m in merges.tolist()[:i]) for i in range(len(merges))]
    assert slots == sum(m[3] for m in merges.tolist())
    assert T.split_items(T.block_items([(0, 8192, 0, 0, 0)], 8192), 32)[1] is None  # 2048 workgroups
    assert T.split_items(T.block_items([(0, 512, 0, 0, 0)], 512), 8)[1] is None     # nothing long


@pytest.mark.gpu
@pytest.mark.parametrize("rows,ctx", [(1, 1024), (70, 1500), (300, 3072), (128, 6144)])
@pytest.mark.parametrize("parts", [2, 3, 8])
def test_parts_of_long_blocks(rows, ctx, parts):
    """Blocks cut into parts against whole ones: the sums are fp32 in another order, then rounded to bf16 once
    on either side (2^-8 of the largest weight's value apart at most)."""
    torch.manual_seed(rows + parts)
    heads, kv = 4, 2
    q = torch.randn(rows, 128 * heads, device=DEV).bfloat16()
    k, v = torch.randn(2, ctx + rows, 128 * kv, device=DEV).bfloat16()
    k[0] *= 3  # a few keys outweigh the rest, so that parts' maxima differ
    items = T.block_items([(0, rows, 0, ctx, 1)], rows)
    want, got = torch.zeros(2, rows + 2, 128 * heads, device=DEV, dtype=torch.bfloat16)
    T.attention_blocks(q, k, v, torch.from_numpy(items).to(DEV), heads, kv, want, k, v)
    out, merges, slot = [], [], 0
    for it in items.tolist():
        merges.append([it[0], it[3] >> 1, slot, parts])
        out += [[*it[:3], it[3] | p << 9 | parts << 13 | slot << 17] for p in range(parts)]
        slot += parts
    T.attention_blocks(q, k, v, torch.tensor(out, dtype=torch.int32, device=DEV), heads, kv, got, k, v,
                       merges=torch.tensor(merges, dtype=torch.int32, device=DEV), slots=slot)
    assert float((got.float() - want.float()).abs().max()) <= 2.0 ** -7 * float(want.float().abs().max())
    assert not got[rows:].any()
    ref = T.ref_attention_chunk(torch.cat([q, q[:, :2 * 128 * kv]], 1), k, v, heads, kv)
    assert float((got[:rows].float() - ref).norm() / ref.norm()) < 2.0 ** -7  # P and the result in bf16


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv", [(8, 2), (3, 1), (4, 4)])
def test_blocks_match_per_sequence_bits(heads, kv):
    """The same tiles in the same order as one launch per sequence: equal bits. Prompts of one and
    several blocks beside chunks whose keys are in other buffers, at contexts that end on a
    block's edge and in its middle."""
    torch.manual_seed(heads)
    lens, past = [128, 384, 256], [(128, 64), (256, 320), (128, 1024)]  # what one launch per sequence takes
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
def test_partial_blocks_match_whole_ones():
    """Lengths and positions of no multiple: each row's bits as in blocks padded to 128 rows, where the
    padding holds other values; nothing past a sequence's rows is written."""
    torch.manual_seed(3)
    heads, kv, w = 4, 2, 8 * 128
    seqs = [(1, 0), (127, 0), (129, 0), (64, 0), (300, 0), (65, 64), (1, 192), (200, 448)]
    rows = sum(n for n, _ in seqs)
    qkv = torch.randn(rows, w, device=DEV).bfloat16()
    k2, v2 = torch.randn(2, sum(c + n for n, c in seqs), 128 * kv, device=DEV).bfloat16()
    plan, want, r, kr = [], [], 0, 0
    for n, c in seqs:
        p = -(-n // 128) * 128
        q = torch.randn(p, w, device=DEV).bfloat16()
        q[:n] = qkv[r:r + n]
        if c:
            k, v = torch.randn(2, c + p, 128 * kv, device=DEV).bfloat16()
            k[:c + n], v[:c + n] = k2[kr:kr + c + n], v2[kr:kr + c + n]
            want.append(T.attention_chunk(q, k, v, heads, kv)[:n])
            plan.append((r, n, kr, c, 1))
            kr += c + n
        else:
            want.append(T.attention_qkv(q, 1, p, heads, kv, out=torch.empty(p, 128 * heads, device=DEV, dtype=torch.bfloat16))[:n])
            plan.append((r, n, r, 0, 0))
        r += n
    out = torch.full((rows + 9, 128 * heads), 5.0, device=DEV, dtype=torch.bfloat16)
    items = torch.from_numpy(T.block_items(plan, rows)).to(DEV)
    T.attention_blocks(qkv, qkv[:, 128 * heads:128 * (heads + kv)], qkv[:, 128 * (heads + kv):], items, heads, kv, out, k2, v2)
    assert torch.equal(out[:rows], torch.cat(want))
    assert bool((out[rows:] == 5).all())


@pytest.mark.gpu
@pytest.mark.parametrize("cache_dtype", [torch.bfloat16, D.FP8])
@pytest.mark.parametrize("lens", [[5, 33, 1], [20] * 9, [700, 400, 31]])
def test_rope_rows_match_padded(lens, cache_dtype):
    """Tokens padded to 128 a prompt whose padding has no rows: the rows and the cache of the padded call."""
    torch.manual_seed(len(lens))
    heads, kv = 4, 2
    total = sum(-(-n // 128) * 128 for n in lens)
    real = sum(lens)
    cos, sin = T.rope_tables(1024, 128, 1e4, DEV)
    pos, slot, rows, at, page, r = np.zeros(total, np.int32), np.full(total, -1, np.int32), np.full(total, -1, np.int32), 0, 1, 0
    for n in lens:
        pos[at:at + n] = np.arange(n)
        slot[at:at + n] = 32 * page + np.arange(n)
        rows[at:at + n] = r + np.arange(n)
        at, page, r = at + -(-n // 128) * 128, page + -(-n // 32), r + n
    pos, slot, rows = (torch.from_numpy(x).to(DEV) for x in (pos, slot, rows))
    qkv = torch.randn(real, (heads + 2 * kv) * 128, device=DEV).bfloat16()
    full = torch.randn(total, (heads + 2 * kv) * 128, device=DEV).bfloat16()
    full[rows >= 0] = qkv
    ca, cb = (torch.zeros(page + 1, kv, 2, 4096, device=DEV).to(cache_dtype) for _ in range(2))
    D.rope_cache_(full, cos, sin, pos, slot, ca, heads, kv)
    D.rope_cache_(qkv, cos, sin, pos, slot, cb, heads, kv, rows=rows)
    assert torch.equal(qkv, full[rows >= 0]) and torch.equal(ca.view(torch.uint8), cb.view(torch.uint8))
    # rows that arrive as partial sums
    parts = torch.randn(4, real, qkv.shape[1], device=DEV)
    whole = parts[0] + parts[1] + parts[2] + parts[3]
    qa, qb = whole.bfloat16(), torch.empty_like(qkv)
    cc, cd = (torch.zeros_like(ca) for _ in range(2))
    D.rope_cache_(qa, cos, sin, pos, slot, cc, heads, kv, rows=rows)
    D.rope_cache_(qb, cos, sin, pos, slot, cd, heads, kv, partials=parts, rows=rows)
    assert torch.equal(qa, qb) and torch.equal(cc.view(torch.uint8), cd.view(torch.uint8))


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


def _prompts(lens):
    """Arguments of a prompt step: prompts padded to 128, each on pages of its own."""
    padded = [-(-n // 128) * 128 for n in lens]
    total, rng = sum(padded), np.random.default_rng(len(lens))
    tok, pos, slot, at, page, starts = np.zeros(total, np.int32), np.zeros(total, np.int32), np.full(total, -1, np.int32), 0, 1, []
    for n, p in zip(lens, padded):
        starts.append(at)
        tok[at:at + n], pos[at:at + n], slot[at:at + n] = rng.integers(0, 1024, n), np.arange(n), 32 * page + np.arange(n)
        at, page = at + p, page + -(-n // 32)
    return (*(torch.from_numpy(a).to(DEV) for a in (tok, pos, slot)), starts, lens, padded)


@pytest.fixture
def normed(monkeypatch):
    """Models whose norm weights are not one, so that a missing or doubled one shows."""
    from kgs.serve import model as M

    class Normed(M.LlamaModel):
        def __init__(self, cfg, **kw):
            super().__init__(cfg, **kw)
            g = torch.Generator(device=DEV).manual_seed(7)
            for t in (*(w[n] for w in self.layers for n in ("ln1", "ln2")), self.norm):
                t.copy_(torch.exp2(torch.rand(t.shape, generator=g, device=DEV) * 4 - 2))

    monkeypatch.setattr(M, "LlamaModel", Normed)
    return M.ServingModel


@pytest.mark.gpu
@pytest.mark.parametrize("lens,ff,fused", [([20, 5], 2048, 48), ([48], 2048, 48), ([49], 2048, 48), ([130, 126], 2048, 48), ([100, 157], 2048, 48),
                                           ([300, 260], 2048, 48), ([20, 5], 2304, 48),  # 2304: no skinny tile of down
                                           ([64], 2048, 128), ([65], 2048, 128), ([257], 2048, 300)])
def test_prefill_by_rows(lens, ff, fused, normed):
    """Either side of the row counts where a prompt step changes its layers: logits and cache of the step
    against float32 layers on the same weights. Sums round to bf16 at other places on either side: a
    few 2^-8 in the 2-norm over two layers."""
    cfg = LlamaConfig(hidden=2048, intermediate=ff, heads=16, kv_heads=4, layers=2, vocab=1024)
    ours, ref = (normed(cfg, device=DEV, backend=b, num_pages=40, max_model_len=1024, fused_max_batch=fused) for b in ("kgs", "ref"))
    args = _prompts(lens)
    got, want = (m.prefill(*args).float() for m in (ours, ref))
    assert got.shape == want.shape == (len(lens), 1024)
    assert float((got - want).norm() / want.norm()) < 0.03
    a, b = ours.cache.data.float(), ref.cache.data.float()
    assert float((a - b).norm() / b.norm()) < 0.02
    assert torch.equal(a == 0, b == 0)  # the same slots written


@pytest.mark.gpu
@pytest.mark.parametrize("lens,kv", [([1], "bf16"), ([20, 5], "bf16"), ([48], "bf16"), ([33], "fp8"), ([64], "bf16"), ([90], "bf16")])
def test_a_prompt_step_repeats_its_bits(lens, kv, normed):
    """The same prompts give the same logits and cached keys every time, whatever order workgroups arrive in."""
    cfg = LlamaConfig(hidden=2048, intermediate=8192, heads=16, kv_heads=4, layers=4, vocab=1024)
    model, args, first = normed(cfg, device=DEV, num_pages=8, max_model_len=256, fused_max_batch=64, kv_cache_dtype=kv), _prompts(lens), None
    for _ in range(40):
        model.cache.data.zero_()
        got = model.prefill(*args).clone(), model.cache.data.view(torch.uint8).clone()
        first = first or got
        assert all(torch.equal(a, b) for a, b in zip(got, first))
