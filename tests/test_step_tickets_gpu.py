"""Tickets of a serving step's decode attention in parts by length: the step's own, cleared by its first launch."""
import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("own_rng")]


@pytest.mark.parametrize("batch", [41, 70])  # the fused layer, the split tiles
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("rows", [True, False])  # by embed_rows, by torch's indexing
def test_a_step_clears_and_leaves_its_tickets(monkeypatch, batch, mixed, rows):
    from kgs.models.llama import LlamaConfig
    from kgs.ops import decode as D
    from kgs.ops import transformer
    from kgs.serve.model import ServingModel

    if not rows:
        monkeypatch.setattr(transformer, "embeds", lambda table: False)
    c = LlamaConfig(hidden=1024, layers=2, heads=8, kv_heads=1, intermediate=512, vocab=512)
    m = ServingModel(c, device="cuda", num_pages=64, max_model_len=2048)
    m.cache.data.normal_()
    i32 = dict(dtype=torch.int32, device="cuda")
    lens = torch.randint(1, 1500, (batch,)).tolist()
    tables = torch.randint(0, 60, (batch, 64), **i32)
    ctx = torch.tensor(lens, **i32)
    tokens, slots = torch.randint(0, 512, (batch,), **i32), torch.full((batch,), -1, **i32)
    seen, real = [], D.paged_decode_attention

    def attention(*a, tickets=None, **kw):
        assert not bool(tickets.any())
        out = real(*a, tickets=tickets, **kw)
        assert not bool(tickets.any())
        seen.append(tickets)
        return out

    def step():
        junk = [torch.full((n,), 7, **i32) for n in (40, 70, 512, 1024)]  # what an allocation finds is not zero
        del junk
        if not mixed:
            return m.decode(tokens, ctx - 1, slots, tables, ctx)
        both = torch.cat([tokens[:32], tokens])
        pos = torch.cat([torch.arange(32, **i32), ctx - 1])
        return m.mixed(both, pos, torch.full((both.numel(),), -1, **i32), [(0, 32, 32, 0, tables[0, :1], True)], tables, ctx)

    monkeypatch.setattr(D, "paged_decode_attention", attention)
    got = step().float()
    assert len(seen) == 2 and seen[0] is seen[1] and seen[0].numel() == batch
    monkeypatch.setattr(D, "paged_decode_attention", real)
    monkeypatch.setattr(D, "part_target", lambda *a: 0)
    want = step().float()
    # sums in another order, rounded to bf16 through two layers
    assert float((got - want).norm() / want.norm()) < 2e-2
