"""The rows that a step starts from (embed_rows in native/kernels/transformer.hip) against torch's indexing and the norm
that it takes the place of."""
import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("own_rng")]
DEV = "cuda"


def table(vocab, cols):
    return torch.randn(vocab, cols, device=DEV).bfloat16()


@pytest.mark.parametrize("cols", [512, 2048, 4096, 8192])
@pytest.mark.parametrize("rows,kept", [(1, None), (3, None), (4, 4), (5, 2), (513, 130), (6, 0)])
def test_rows_norm_squares_and_zeros(cols, rows, kept):
    from kgs.ops.transformer import add_rmsnorm, embed_rows

    emb, w = table(77, cols), torch.randn(cols, device=DEV).bfloat16()
    tokens = torch.randint(0, 77, (rows,), device=DEV, dtype=torch.int32)
    tokens[0] = 76
    pos, slot = (torch.randint(-1, 1 << 20, (rows,), device=DEV, dtype=torch.int32) for _ in range(2))
    keep = None if kept is None else torch.randperm(rows, device=DEV)[:kept].int()
    at = slice(None) if keep is None else keep.long()
    want = emb[tokens.long()[at]]
    ss = torch.full((want.shape[0],), 9.0, device=DEV)
    z1, z2 = torch.ones(2, 8, 7, dtype=torch.int64, device=DEV), torch.ones(1001, dtype=torch.int32, device=DEV)
    x, y, p, s = embed_rows(emb, tokens, w, 1e-5, keep, ss, pos, slot, (z1, z2[:1000]))
    assert torch.equal(x, want) and torch.equal(p, pos[at]) and torch.equal(s, slot[at])
    assert torch.equal(y, add_rmsnorm(want.clone(), None, w, 1e-5) if want.shape[0] else want)
    exact = want.double().pow(2).sum(-1)
    assert float((ss - exact).abs().max() if want.shape[0] else 0) <= cols * 2.0 ** -24 * float(exact.max() if want.shape[0] else 1)
    assert not z1.any() and not z2[:1000].any() and int(z2[1000]) == 1
    x, y, p, s = embed_rows(emb, tokens.long(), None, keep=keep)  # other integers, nothing else wanted
    assert torch.equal(x, want) and y is None and p is None and s is None


def test_numbers_off_the_table():
    """Below zero from the end, as torch's; past either end NaN and no read outside the table."""
    from kgs.ops.transformer import embed_rows

    emb = table(10, 512)
    tokens = torch.tensor([-1, -10, -11, 9, 10, 2 ** 31 - 1, -2 ** 31, 0], device=DEV)
    x, y, _, _ = embed_rows(emb, tokens, torch.ones(512, device=DEV).bfloat16())
    bad = [2, 4, 5, 6]
    assert bool(x[bad].isnan().all()) and bool(y[bad].isnan().all())
    assert torch.equal(x[[0, 1, 3, 7]], emb[[9, 0, 9, 0]])
    assert bool(embed_rows(emb, torch.tensor([2 ** 32 + 1], device=DEV))[0].isnan().all())


def test_what_it_refuses_and_replays():
    from kgs.ops.transformer import embed_rows, embeds

    emb, tok = table(10, 512), torch.zeros(4, dtype=torch.int32, device=DEV)
    assert not embeds(table(10, 520)) and not embeds(emb.float()) and not embeds(emb.cpu()) and not embeds(table(4, 8704))
    for bad in (lambda: embed_rows(table(10, 520), tok), lambda: embed_rows(emb, tok.cpu()), lambda: embed_rows(emb, tok, emb[0].float()),
                lambda: embed_rows(emb, tok, squares=torch.zeros(3, device=DEV)), lambda: embed_rows(emb, tok, positions=tok[:2]),
                lambda: embed_rows(emb, tok, keep=tok.long()), lambda: embed_rows(emb, tok, zeros=(torch.zeros(3, device=DEV).bfloat16(),))):
        with pytest.raises(ValueError):
            bad()
    z = torch.ones(5, device=DEV)
    graph = torch.cuda.CUDAGraph()
    embed_rows(emb, tok)
    with torch.cuda.graph(graph):
        x = embed_rows(emb, tok, zeros=(z,))[0]
    for t in (3, 7, 1):
        tok.fill_(t)
        z.fill_(1.0)
        graph.replay()
        assert torch.equal(x, emb[[t] * 4]) and not z.any()
        torch.cuda.synchronize()


@pytest.mark.parametrize("batch", [5, 70])  # the fused layer, the split tiles
def test_steps_take_what_indexing_took(batch):
    """Tokens in host memory, positions and slots of a longer batch, prompts' positions and slots from columns of a matrix."""
    from kgs.models.llama import LlamaConfig
    from kgs.serve.model import ServingModel

    m = ServingModel(LlamaConfig(hidden=1024, layers=1, heads=8, kv_heads=1, intermediate=512, vocab=512), device="cuda", num_pages=64,
                     max_model_len=512)
    i32 = dict(dtype=torch.int32, device=DEV)
    tokens, pos = torch.randint(0, 512, (batch,), **i32), torch.zeros(batch, **i32)
    slots, tables, ctx = torch.full((batch,), -1, **i32), torch.zeros(batch, 1, **i32), torch.ones(batch, **i32)
    want = m.decode(tokens, pos, slots, tables, ctx).float()

    def same(got):
        # the fused layer adds its rows' squares in the order of arrival
        assert float((got.float() - want).norm() / want.norm()) < 1e-2

    same(m.decode(tokens.cpu(), pos, slots, tables, ctx))
    same(m.decode(tokens.long(), pos, slots, tables, ctx))
    if batch < 48:
        same(m.decode(tokens, torch.cat([pos, pos]), torch.cat([slots, slots]), tables, ctx))
        n = 32
        prompt, at, to = torch.randint(0, 512, (n,), **i32), torch.arange(n, **i32), torch.arange(n, **i32) + 32
        cols = torch.stack([at, to], 1)
        assert not cols[:, 0].is_contiguous()
        assert torch.equal(m.prefill(prompt, cols[:, 0], cols[:, 1], [0], [20], [32]), m.prefill(prompt, at, to, [0], [20], [32]))
