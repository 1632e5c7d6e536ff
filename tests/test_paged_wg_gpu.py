"""Decode attention by workgroups (paged_wg in native/kernels/decode.hip) where its parts meet:
one token, page and wave borders, more parts than pages, one and sixteen query heads per key
head, contexts of very different lengths, e4m3 pages, replays from a hipGraph."""
import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu
DEV = "cuda"


def setup(lens, hkv, group, fp8=False, seed=0):
    from kgs.ops import decode as D

    g = torch.Generator(device=DEV).manual_seed(seed)
    need = [math.ceil(n / 32) for n in lens]
    cache = torch.randn(sum(need) + 1, hkv, 2, 4096, device=DEV, generator=g).to(D.FP8 if fp8 else torch.bfloat16)
    ids = 1 + torch.randperm(sum(need), device=DEV, generator=g).int()
    tables = torch.zeros(len(lens), max(need) + 3, dtype=torch.int32, device=DEV)
    at = 0
    for i, n in enumerate(need):
        tables[i, :n] = ids[at:at + n]
        at += n
    q = (2 * torch.randn(len(lens), (group + 2) * hkv * 128, device=DEV, generator=g)).bfloat16()
    return q, cache, tables, torch.tensor(lens, dtype=torch.int32, device=DEV)


def run(q, cache, tables, ctx, heads, hkv, nsplit, out):
    from kgs.ops import _lib
    from kgs.ops import decode as D

    ws = D._attn_workspace(q.shape[0], heads, hkv, nsplit, q.device)
    rc = _lib.lib().kgs_paged_decode_wg(q.data_ptr(), cache.data_ptr(), tables.data_ptr(), ctx.data_ptr(), out.data_ptr(),
                                        *(None if t is None else t.data_ptr() for t in ws), q.shape[0], heads, hkv, 128,
                                        tables.shape[1], nsplit, q.stride(0), out.stride(0), 128 ** -0.5,
                                        int(cache.dtype == D.FP8), _lib.stream_handle(q.device))
    assert rc == 0


# weights and values are bf16 (2^-8 each), so a row moves by at most their product's share of |v| < 6
TOL = 3e-2


@pytest.mark.parametrize("hkv,group", [(8, 4), (1, 16), (4, 1), (2, 7)])
@pytest.mark.parametrize("nsplit", [1, 2, 5])
@pytest.mark.parametrize("fp8", [False, True])
def test_parts_and_lengths(hkv, group, nsplit, fp8):
    from kgs.ops import decode as D

    lens = [1, 31, 32, 33, 256, 257, 300, 2200]
    q, cache, tables, ctx = setup(lens, hkv, group, fp8)
    want = D.ref_paged_decode(q, cache, tables, ctx, hkv * group, hkv)
    out = torch.full((len(lens) + 1, hkv * group * 128), 7.0, dtype=torch.bfloat16, device=DEV)
    for _ in range(2):  # the merge leaves its tickets at zero
        run(q, cache, tables, ctx, hkv * group, hkv, nsplit, out[:len(lens)])
        assert float((out[:len(lens)].float() - want).abs().max()) < TOL
    assert bool((out[-1] == 7).all())


def test_an_empty_context_gives_zeros_and_a_graph_replays():
    from kgs.ops import decode as D

    q, cache, tables, ctx = setup([40, 500, 90, 1000], 8, 4)
    ctx[2] = 0
    eager = D.paged_decode_attention(q, cache, tables, ctx, 32, 8)
    assert bool((eager[2] == 0).all())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = D.paged_decode_attention(q, cache, tables, ctx, 32, 8)
    for _ in range(3):
        out.zero_()
        graph.replay()
        D.paged_decode_attention(q, cache, tables, ctx, 32, 8)
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


@pytest.mark.parametrize("batch,kv,pages", [(1, 8, 1), (1, 8, 32), (1, 1, 4096), (16, 8, 128), (64, 8, 64), (300, 8, 16)])
def test_split_rule_stays_in_its_bounds(batch, kv, pages):
    from kgs.ops.decode import workgroup_splits

    n = workgroup_splits(batch, kv, pages)
    assert 1 <= n <= max(1, pages // 8) and (n == 1 or (n - 1) * batch * kv < 512)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("lens,kv,pages", [([512], 8, 16), ([1, 0, 33, 512], 8, 16), ([70] * 8, 4, 16), ([992], 8, 31), ([1024], 8, 32), ([40, 513], 4, 32), ([2000], 8, 63)])
def test_shorter_parts(lens, kv, pages, fp8):
    """Few pairs in tables of 16 to 63 pages: parts with no page, with one and with all of theirs."""
    from kgs.ops import decode as D

    b = len(lens)
    parts, waves = D.shorter_parts(b, kv, pages, 4 if fp8 else 8, fp8)
    if pages < 32 or not fp8:
        assert (parts, waves) == (4 if pages < 32 else 8, 4) and D.shorter_parts(33, 1, pages, 8, fp8)[1] == 8
    g = torch.Generator(device=DEV).manual_seed(pages)
    cache = torch.randn(70, kv, 2, 4096, device=DEV, generator=g).to(D.FP8 if fp8 else torch.bfloat16)
    tables, ctx = torch.randint(0, 70, (b, pages), generator=g, device=DEV, dtype=torch.int32), torch.tensor(lens, device=DEV, dtype=torch.int32)
    q = (2 * torch.randn(b, 4 * kv * 128, device=DEV, generator=g)).bfloat16()
    got = D.paged_decode_attention(q, cache, tables, ctx, 4 * kv, kv)
    want = D.ref_paged_decode(q, cache, tables, ctx.clamp(min=1), 4 * kv, kv)
    want[ctx == 0] = 0
    assert float((got.float() - want).abs().max()) < TOL


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("groups", [1, 639, 640, 1023, 1024, 1151, 1152, 1535, 1536, 2047, 2048, 8192])
@pytest.mark.parametrize("pages", [1, 2, 3, 4, 5, 8, 9, 16, 17, 4096])
def test_wave_rule(fp8, groups, pages):
    """Narrow tables by few waves, the fewer the more pairs there are; everything else by as many as elsewhere."""
    from kgs.ops.decode import workgroup_waves

    w, most = workgroup_waves(groups, pages, fp8), 4 if fp8 else 8
    assert w in ((1, 2, 4) if fp8 else (1, 2, 4, 8))
    assert w == most or pages <= (16 if fp8 else 8)
    assert w <= workgroup_waves(groups, pages + 1, fp8) and w >= workgroup_waves(groups + 1, pages, fp8)
    assert w == 1 if pages == 1 and (groups >= 640 or not fp8) else w > 1 or groups >= (1152 if pages > 2 else 1024)
    assert w == 1 or not (fp8 and pages <= 2 and groups >= 1024)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("pages", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("batch", [5, 79, 80, 127, 128, 144, 256])
def test_few_waves_on_narrow_tables(batch, pages, fp8):
    """Either side of each border of the rule, contexts of every length that the table holds."""
    from kgs.ops import decode as D

    g = torch.Generator(device=DEV).manual_seed(pages)
    ctx = torch.randint(1, 32 * pages + 1, (batch,), generator=g, device=DEV, dtype=torch.int32)
    ctx[0], ctx[1], ctx[2] = 32 * pages, 1, 0
    cache = torch.randn(50, 8, 2, 4096, device=DEV, generator=g).to(D.FP8 if fp8 else torch.bfloat16)
    tables = torch.randint(0, 50, (batch, pages), generator=g, device=DEV, dtype=torch.int32)
    q = (2 * torch.randn(batch, 16 * 128, device=DEV, generator=g)).bfloat16()
    got = D.paged_decode_attention(q, cache, tables, ctx, 16, 8)
    some = [0, 1, 2, *range(3, batch, 17), batch - 1]
    want = D.ref_paged_decode(q[some], cache, tables[some].contiguous(), ctx[some].clamp(min=1), 16, 8)
    want[2] = 0
    assert float((got[some].float() - want).abs().max()) < TOL


@pytest.mark.parametrize("fp8,waves", [(False, 2), (False, 4), (True, 2)])
@pytest.mark.parametrize("nsplit", [1, 3])
def test_few_waves_in_parts(fp8, waves, nsplit):
    from kgs.ops import _lib
    from kgs.ops import decode as D

    lens, hkv = [1, 33, 64, 65, 129, 900, 2200], 4
    q, cache, tables, ctx = setup(lens, hkv, 4, fp8)
    out = torch.full((len(lens), 16 * 128), 7.0, dtype=torch.bfloat16, device=DEV)
    ws = D._attn_workspace(len(lens), 16, hkv, nsplit, q.device)

    def go(w):
        return _lib.lib().kgs_paged_decode_wg_ex(q.data_ptr(), cache.data_ptr(), tables.data_ptr(), ctx.data_ptr(), out.data_ptr(),
                                                 *(None if t is None else t.data_ptr() for t in ws), len(lens), 16, hkv, 128, tables.shape[1],
                                                 nsplit, q.stride(0), out.stride(0), 128 ** -0.5, int(fp8), w, _lib.stream_handle(q.device))

    assert go(waves) == 0
    assert float((out.float() - D.ref_paged_decode(q, cache, tables, ctx, 16, hkv)).abs().max()) < TOL
    assert go(3) != 0 and go(8 if fp8 else 1) != 0  # no such kernels


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hkv,group", [(8, 4), (1, 16), (4, 1)])
@pytest.mark.parametrize("batch,target", [(1, 7), (9, 1), (9, 3), (64, 40), (65, 40), (128, 300)])
def test_parts_that_follow_the_lengths(batch, target, hkv, group, fp8):
    """One part each, parts of one round, more than eight of a sequence, empty contexts, both sides of 64 sequences; rows and
    tables past the batch stay as they are, and tickets end at zero."""
    from kgs.ops import _lib
    from kgs.ops import decode as D

    g = torch.Generator(device="cpu").manual_seed(batch)
    lens = torch.randint(1, 400, (batch,), generator=g).tolist()
    lens[0], lens[-1] = 2200, 1 if batch > 1 else 2200
    q, cache, tables, ctx = setup(lens, hkv, group, fp8)
    if batch > 2:
        ctx[2] = 0
    heads = hkv * group
    want = D.ref_paged_decode(q, cache, tables, ctx.clamp(min=1), heads, hkv)
    out = torch.full((batch + 1, heads * 128), 7.0, dtype=torch.bfloat16, device=DEV)
    rows = batch + target
    po, pml = torch.full(((rows * heads + 1) * 128,), 7.0, device=DEV), torch.full((rows * heads * 2 + 2,), 7.0, device=DEV)
    cnt = torch.zeros(batch * hkv, dtype=torch.int32, device=DEV)
    for least in (1, 8, 64):
        rc = _lib.lib().kgs_paged_decode_wg_bal(q.data_ptr(), cache.data_ptr(), tables.data_ptr(), ctx.data_ptr(), out.data_ptr(),
                                                po.data_ptr(), pml.data_ptr(), cnt.data_ptr(), batch, heads, hkv, 128, tables.shape[1],
                                                target, least, q.stride(0), out.stride(0), 128 ** -0.5, int(fp8),
                                                _lib.stream_handle(q.device))
        assert rc == 0
        got = out[:batch].float()
        if batch > 2:
            assert bool((got[2] == 0).all())
            got[2] = want[2]
        assert float((got - want).abs().max()) < TOL
        assert bool((out[-1] == 7).all()) and bool((po[-128:] == 7).all()) and bool((pml[-2:] == 7).all()) and not bool(cnt.any())


def test_length_rule_has_room_for_its_parts():
    from kgs.ops.decode import length_parts

    for batch in (1, 2, 3, 31, 32, 64, 128, 129):
        for kv in (1, 4, 8, 300):
            for fp8 in (False, True):
                n = length_parts(batch, kv, 64, 4 if fp8 else 8, fp8)
                assert (n > 0) == (2 < batch <= 128) and n * kv <= max(384, kv)
                assert length_parts(batch, kv, 63, 4 if fp8 else 8, fp8) == 0 == length_parts(batch, kv, 64, 2, fp8)


@pytest.mark.parametrize("batch,kv,target", [(3, 8, 24), (19, 8, 24), (20, 8, 48), (153, 1, 0), (38, 4, 48), (39, 4, 96), (128, 8, 48), (100, 4, 96), (5, 300, 1)])
@pytest.mark.parametrize("fp8", [False, True])
def test_parts_by_the_number_of_pairs(batch, kv, target, fp8):
    from kgs.ops.decode import length_parts

    assert length_parts(batch, kv, 64, 4 if fp8 else 8, fp8) == target


@pytest.mark.parametrize("batch,kv,pages,parts", [(5, 8, 64, False), (5, 8, 127, False), (5, 8, 128, True), (41, 1, 64, True), (11, 4, 64, True), (3, 1, 4096, True)])
def test_few_pairs_on_narrow_tables_keep_equal_parts(batch, kv, pages, parts):
    from kgs.ops import decode as D

    assert bool(D.part_tickets(batch, kv, pages, False)) == parts
    lens = [32 * pages - 5] + [70] * (batch - 1)
    q, cache, tables, ctx = setup(lens, kv, 2)
    tables = tables[:, :pages].contiguous()
    got = D.paged_decode_attention(q, cache, tables, ctx, 2 * kv, kv).float()
    assert float((got - D.ref_paged_decode(q, cache, tables, ctx, 2 * kv, kv)).abs().max()) < TOL


def test_parts_keep_their_scratch_to_the_call(monkeypatch):
    """Batches that had no split before their parts followed the lengths shared nothing with other calls, nor do they now: steps
    of different lengths on two streams, and between a graph's replays, with tickets given and without."""
    from kgs.ops import decode as D

    monkeypatch.setattr(D, "_attn_workspace", lambda *a: pytest.fail("workspace of the whole GPU"))
    g = torch.Generator().manual_seed(1)
    sets = []
    for _ in range(4):
        lens = torch.randint(1, 700, (64,), generator=g).tolist()
        lens[5] = 2040
        sets.append(setup(lens, 8, 2, seed=len(sets)))
    assert D.part_tickets(64, 8, sets[0][2].shape[1], False) == 512
    want = [D.paged_decode_attention(*s, 16, 8) for s in sets]
    for w, s in zip(want, sets):
        assert float((w.float() - D.ref_paged_decode(*s, 16, 8)).abs().max()) < TOL
    tickets = [torch.zeros(512, dtype=torch.int32, device=DEV) for _ in sets]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    got = []
    for n in range(10):
        for i, s in enumerate(sets):
            with torch.cuda.stream(streams[i % 2]):
                got.append((i, D.paged_decode_attention(*s, 16, 8, tickets=tickets[i % 2] if n % 2 else None)))
    torch.cuda.synchronize()
    assert all(torch.equal(o, want[i]) for i, o in got) and not any(bool(t.any()) for t in tickets)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = D.paged_decode_attention(*sets[0], 16, 8)
    for _ in range(4):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        with torch.cuda.stream(streams[0]):
            other = D.paged_decode_attention(*sets[1], 16, 8)
        torch.cuda.synchronize()
        assert torch.equal(out, want[0]) and torch.equal(other, want[1])
    for bad in (tickets[0][:511], tickets[0].long(), tickets[0].cpu(), torch.zeros(1024, dtype=torch.int32, device=DEV)[::2]):
        with pytest.raises(ValueError):
            D.paged_decode_attention(*sets[0], 16, 8, tickets=bad)
