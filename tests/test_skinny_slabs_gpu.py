"""Skinny products in K slices (native/kernels/decode_slabs.hip) against the plain product in float64, and the hyper-connection step that adds the slices."""
import pytest
import torch

from kgs.ops import decode as D
from kgs.ops.activation import Gate
from kgs.ops.hyper import hyper_step

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("own_rng")]


def _operands(m, n, k, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(m, k + 8, generator=g, device="cuda").bfloat16()[:, :k]  # rows further apart than they are long
    return x, (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).bfloat16()


# the shortest slice (one round of the weights' ring), one chunk more, many; one and two tiles a wave; column tiles full, of one row and short
@pytest.mark.parametrize("n,k", ((64, 128), (64, 256), (1024, 1024), (2048, 2048), (2048, 8192), (192, 384), (4096, 896), (4224, 2048)))
@pytest.mark.parametrize("m", (1, 16, 17, 32, 33, 64, 65, 96))
def test_slices_add_to_the_product(n, k, m):
    x, w = _operands(m, n, k)
    r, ns = D.slab_split(m, n, k)
    got = D.skinny_slabs(x, D.PackedWeight(w))
    assert got.shape == (ns, m, n) and k % (128 * ns) == 0 and n % (64 * r) == 0
    ks = k // ns
    for i in range(ns):
        ref = x[:, i * ks:(i + 1) * ks].double() @ w[:, i * ks:(i + 1) * ks].double().T
        # fp32 sums of ks products of bf16: the roundings of ks additions, on average their root
        assert float((got[i].double() - ref).abs().max()) <= 2.0 ** -24 * ks * float(ref.abs().max())


# each side of the lines between 128-row strips in eight slices and 64-row ones in four, and between eight slices and four of a short K
@pytest.mark.parametrize("m,n,k,split", ((1, 4096, 2048, (1, 4)), (96, 4096, 8192, (1, 4)), (96, 4096, 12288, (2, 8)), (33, 8192, 8192, (2, 4)), (97, 4096, 4096, (1, 4)),
                                         (128, 4096, 16384, (2, 8)), (32, 2048, 2048, (1, 8)), (33, 2048, 2048, (1, 4)), (128, 2048, 1024, (1, 4)), (33, 2048, 4096, (1, 8)), (40, 1024, 512, (1, 4))))
def test_fewer_slices(m, n, k, split):
    x, w = _operands(m, n, k)
    rule, slabs = (D.slab_split, D.skinny_slabs) if m <= 96 else (D.wide_split, D.wide_slabs)
    assert rule(m, n, k) == split and (m > 96 or D.slabs_fill(m, n, k) or (n, k) == (1024, 512))
    got, ks, ref = slabs(x, D.PackedWeight(w)), k // split[1], x.double() @ w.double().T
    # fp32 sums of ks products of bf16 in each of the slices: the roundings of ks additions, on average their root
    assert got.shape == (split[1], m, n) and float((got.double().sum(0) - ref).abs().max()) <= 2.0 ** -24 * ks * float(ref.abs().max())


def test_what_slices_do_not_take():
    for m, n, k in ((0, 2048, 2048), (97, 2048, 2048), (8, 2080, 2048), (8, 2048, 2080)):
        assert D.slab_split(m, n, k) is None
    x, w = _operands(4, 128, 256)
    for pw in (D.PackedWeight(w, swiglu=True), D.PackedWeight(w, fp8=True)):
        with pytest.raises(ValueError):
            D.skinny_slabs(x, pw)
    for m, n, k in ((0, 2048, 2048), (97, 2048, 2048), (40, 2080, 2048), (40, 2048, 2080)):
        assert D.slab_rows_tiles(m, n, k) is None
    with pytest.raises(ValueError):
        D.skinny_rows(x, D.PackedWeight(w, fp8=True))
    with pytest.raises(ValueError):
        D.skinny_rows(x, D.PackedWeight(w), sq=torch.ones(3, device="cuda"))


# short and deep rings (the latter from 33 rows and 192 strips of 128 rows on), the latter's least and one round more
@pytest.mark.parametrize("n,k", ((64, 128), (1024, 384), (16384, 256), (24576, 256), (24576, 512), (24576, 384), (24704, 1024)))
@pytest.mark.parametrize("m", (1, 16, 17, 32, 33, 64, 65, 96))
def test_whole_products_and_gates(n, k, m):
    x, w = _operands(m, n, k, 1)
    ref = x.double() @ w.double().T

    def close(got, want, factors=1):  # one rounding to bf16, and fp32 sums' errors for each factor
        assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2e-5 * factors * want.abs().max()).all())

    close(D.skinny_rows(x, D.PackedWeight(w)), ref)
    sq = x.float().pow(2).sum(1)
    normed = ref * torch.rsqrt(x.double().pow(2).mean(1, keepdim=True) + 1e-3)
    close(D.skinny_rows(x, D.PackedWeight(w), sq, 1e-3), normed)
    g, u = normed.chunk(2, 1)
    close(D.skinny_rows(x, D.PackedWeight(w, swiglu=True), sq, 1e-3), torch.nn.functional.silu(g) * u, 4)
    close(D.skinny_rows(x, D.PackedWeight(w, swiglu=True, act="gelu_tanh"), sq, 1e-3), torch.nn.functional.gelu(g, approximate="tanh") * u, 4)
    c, v = g.clamp(max=0.5), u.clamp(-0.5, 0.5)
    close(D.skinny_rows(x, D.PackedWeight(w, swiglu=True, act=Gate("clamped", 0.5)), sq, 1e-3), c * torch.sigmoid(1.702 * c) * (v + 1), 4)


def test_weights_of_more_than_31_bits_of_values():
    """An LM head of 2.15e9 values: its first, middle and last strips."""
    from kgs.ops.linear import Projection

    m, n, k = 33, 131200, 16384
    x, w = _operands(m, 128, k, 3)
    wide = w.repeat(n // 128, 1)
    wide[-1] *= 2
    ref = (x.double() @ w.double().T).repeat(1, n // 128)
    ref[:, -1] *= 2
    p = Projection(wide)
    assert n * k > 1 << 31 and D.slab_rows_tiles(m, n, k) == 2
    for got in (D.skinny_rows(x, p.packed), p(x)):
        assert bool(((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2e-5 * ref.abs().max()).all())


@pytest.mark.parametrize("heads,kv,k", ((32, 8, 4096), (16, 4, 2048), (8, 1, 128), (2, 1, 1024)))  # 4, 4, 1 and 4 slices
@pytest.mark.parametrize("m", (33, 96))
def test_rotation_of_slices_as_of_the_whole_product(heads, kv, k, m):
    from kgs.ops.transformer import rope_tables

    x, w = _operands(m, (heads + 2 * kv) * 128, k, 2)
    cos, sin = rope_tables(256, 128, 10000.0, "cuda")
    pos, slots = torch.arange(m, dtype=torch.int32, device="cuda") * 7 % 250, torch.randperm(256, device="cuda")[:m].int()
    slots[5] = -1
    caches = [D.PagedKVCache(1, 8, kv, "cuda") for _ in range(2)]
    pw = D.PackedWeight(w, rope=(heads, kv))
    sq = x.float().pow(2).sum(1)
    parts = D.skinny_slabs(x, pw)
    got = D.rope_cache_packed(parts, sq, pw, 1e-5, {"cos": cos, "sin": sin, "positions": pos, "slots": slots, "cache": caches[0].layer(0)})
    total = parts[0].clone()
    for p in parts[1:]:
        total += p
    total *= torch.rsqrt(sq[:, None] * (1.0 / k) + 1e-5)
    want = torch.empty_like(total)
    want[:, D.rope_rows(pw.n, heads, kv).cuda()] = total
    want = want.bfloat16()
    D.rope_cache_(want, cos, sin, pos, slots, caches[1].layer(0), heads, kv)
    # v_rsq's last bit before the rounding to bf16
    assert float((got.float() - want.float()).abs().max()) <= 2.0 ** -7 * float(want.float().abs().max())
    assert float((got.float() - want.float()).norm() / want.float().norm()) < 1e-3
    assert float((caches[0].data.float() - caches[1].data.float()).norm() / caches[1].data.float().norm()) < 1e-3
    assert torch.equal(caches[0].data == 0, caches[1].data == 0)


# one slice and eight, one and two tiles a wave, the last column tile full and of one row
@pytest.mark.parametrize("n,k", ((64, 128), (2048, 2048), (4096, 384), (4224, 2048), (24576, 256)))
@pytest.mark.parametrize("m", (97, 112, 113, 128))
def test_wide_slices_and_products(n, k, m):
    x, w = _operands(m, n, k, 3)
    ns, pw = D.wide_split(m, n, k)[1], D.PackedWeight(w)
    ref = x.double() @ w.double().T
    got = D.wide_slabs(x, pw)
    assert got.shape == (ns, m, n)
    # as test_slices_add_to_the_product, whose bound holds for each slice
    assert float((got.double().sum(0) - ref).abs().max()) <= 2.0 ** -24 * k * float(ref.abs().max())
    y = D.wide_rows(x, pw)
    assert bool(((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2e-5 * ref.abs().max()).all())
    sq = x.float().pow(2).sum(1)
    normed = ref * torch.rsqrt(x.double().pow(2).mean(1, keepdim=True) + 1e-3)
    assert bool(((D.wide_rows(x, pw, sq, 1e-3).double() - normed).abs() <= 2.0 ** -8 * normed.abs() + 2e-5 * normed.abs().max()).all())


# five, six and seven waves of one tile: whole strips, and strips whose last waves have no tile (22016, 17408, 25088)
@pytest.mark.parametrize("n,k", ((5120, 1024), (6144, 2048), (28672, 128), (22016, 384), (17408, 256), (25088, 128)))
@pytest.mark.parametrize("m", (1, 17, 48, 65, 97, 128))
def test_strips_that_fill_the_cus(n, k, m):
    x, w = _operands(m, n, k, 4)
    ref, pw = x.double() @ w.double().T, D.PackedWeight(w)
    rule, slabs, rows = (D.slab_split, D.skinny_slabs, D.skinny_rows) if m <= 96 else (D.wide_split, D.wide_slabs, D.wide_rows)
    got = slabs(x, pw)
    assert got.shape == (rule(m, n, k)[1], m, n)
    assert float((got.double().sum(0) - ref).abs().max()) <= 2.0 ** -24 * k * float(ref.abs().max())

    def close(got, want, factors=1):  # as test_whole_products_and_gates
        assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2e-5 * factors * want.abs().max()).all())

    close(rows(x, pw), ref)
    if m <= 96:
        g, u = ref.chunk(2, 1)
        close(D.skinny_rows(x, D.PackedWeight(w, swiglu=True)), torch.nn.functional.silu(g) * u, 4)


@pytest.mark.parametrize("rows", (97, 128))
@pytest.mark.parametrize("inter", (1024, 8192))  # gate and up by the library and by the gate kernel
def test_layers_of_wide_slices_as_the_others(rows, inter):
    from kgs.models.llama import LlamaConfig
    from kgs.serve.model import ServingModel

    m = ServingModel(LlamaConfig(hidden=2048, layers=2, heads=16, kv_heads=4, intermediate=inter, vocab=12288), device="cuda", num_pages=256, max_model_len=1024)
    m.cache.data.normal_()
    assert m._wide(rows) and not m._wide(96) and not m._wide(129) and D.head_pays(rows, 12288, 2048) and not m._slab_prompts(rows)
    m._slab_prompts = lambda rows: m._wide(rows)  # prompts as well, which the host bounds with layers of so few weights
    i32 = dict(dtype=torch.int32, device="cuda")
    ctx, tokens, slots = torch.randint(1, 300, (rows,), **i32), torch.randint(0, 512, (rows,), **i32), torch.full((rows,), -1, **i32)
    tables = torch.stack([torch.randperm(255, device="cuda")[:16].int() + 1 for _ in range(rows)])
    flat, pos = torch.randint(0, 512, (128,), **i32), torch.arange(128, **i32)
    where = torch.where(pos < rows, pos + 32, -1).int()

    def both():
        m.cache.data[:, 1:32].zero_()
        logits = m.prefill(flat, pos, where, [0], [rows], [128])
        return m.decode(tokens, ctx - 1, slots, tables, ctx).float(), logits.float(), m.cache.data.float()

    got, again = both(), both()
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    m._wide = lambda rows: False
    for a, b in zip(got, both()):
        assert float((a - b).norm() / b.norm()) < 2e-2  # sums in another order, rounded to bf16 through two layers


@pytest.mark.parametrize("cols", (2048, 4096, 6144, 8192))
@pytest.mark.parametrize("parts", (1, 2, 4, 8, 16))
def test_residual_add_of_slices_and_its_squares(parts, cols):
    from kgs.ops.transformer import splitk_add_squares

    g = torch.Generator(device="cuda").manual_seed(cols)
    p = torch.randn(parts, 5, cols, generator=g, device="cuda")
    x = torch.randn(5, cols, generator=g, device="cuda").bfloat16()
    total = p[0].clone()
    for q in p[1:]:
        total += q
    want = (x.float() + total).bfloat16()
    sq = splitk_add_squares(p, x)
    assert torch.equal(x, want)
    assert torch.allclose(sq.double(), want.double().pow(2).sum(1), rtol=1e-6)


@pytest.mark.parametrize("cols", (2048, 8192))
def test_squares_are_sums_rounded_once(cols):
    from kgs.ops.transformer import splitk_add_squares

    g = torch.Generator(device="cuda").manual_seed(cols)
    x = torch.randn(400, cols, generator=g, device="cuda").bfloat16()
    sq = splitk_add_squares(torch.randn(2, 400, cols, generator=g, device="cuda"), x)
    want = x.double().pow(2).sum(1)
    # the rounding to fp32 and, averaged over 256 chunks and more of eight values, theirs
    assert float((sq.double() / want - 1).abs().max()) <= 1.25 * 2.0 ** -24


@pytest.mark.parametrize("rows", (33, 48, 49, 64, 96))
@pytest.mark.parametrize("wide", (False, True))  # gate and up of a product's two tiles a wave
def test_layers_of_slices_as_the_others(rows, wide):
    from kgs.models.llama import LlamaConfig
    from kgs.serve.model import ServingModel

    c = LlamaConfig(hidden=2048, layers=2, heads=16, kv_heads=4, intermediate=12544 if wide else 1024, vocab=512)
    m = ServingModel(c, device="cuda", num_pages=256, max_model_len=1024)
    m.cache.data.normal_()
    assert m._slabs(rows) and not m._slabs(32) and not m._slabs(97)
    i32 = dict(dtype=torch.int32, device="cuda")
    ctx = torch.randint(1, 300, (rows,), **i32)
    tables = torch.stack([torch.randperm(255, device="cuda")[:16].int() + 1 for _ in range(rows)])
    tokens, slots = torch.randint(0, 512, (rows,), **i32), torch.full((rows,), -1, **i32)
    n = [rows // 2, rows - rows // 2]
    starts, padded = [0, 128], [128, 128]
    flat = torch.randint(0, 512, (256,), **i32)
    pos = torch.cat([torch.arange(128, **i32)] * 2)
    where = torch.cat([torch.where(torch.arange(128, device="cuda") < k, torch.arange(128, device="cuda") + o, -1) for k, o in zip(n, (32, 512))]).int()

    def both():
        m.cache.data[:, 1:32].zero_()
        logits = m.prefill(flat, pos, where, starts, n, padded)
        return m.decode(tokens, ctx - 1, slots, tables, ctx).float(), logits.float(), m.cache.data.float()

    got, again = both(), both()
    assert all(torch.equal(a, b) for a, b in zip(got, again))  # both steps' bits repeat
    m._slabs = m._slab_prompts = lambda rows: False
    for a, b in zip(got, both()):
        assert float((a - b).norm() / b.norm()) < 2e-2  # sums in another order, rounded to bf16 through two layers


@pytest.mark.parametrize("width", (64, 1023, 1028, 2048, 2052, 4096, 4100))  # both kernels' edges and rows that 16-byte loads cannot read
@pytest.mark.parametrize("parts", (1, 5, 8, 9))
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float32))
def test_step_adds_parts_as_it_takes_their_sum(dtype, parts, width):
    t, s = 7, 4
    g = torch.Generator(device="cuda").manual_seed(width)
    rnd = lambda *sh: torch.randn(*sh, generator=g, device="cuda")  # noqa: E731
    y = rnd(parts, t, width)
    args = (rnd(s, s), rnd(s), rnd(s), rnd(width))
    total = y[0].clone()
    for p in y[1:]:
        total += p
    a = rnd(t, s, width)
    b = a.clone()
    want = hyper_step(a, total.to(dtype), *args, 1e-5, ld=width + 4)
    got = hyper_step(b, y, *args, 1e-5, dtype=dtype, ld=width + 4)
    assert torch.equal(a, b) and torch.equal(got, want)


@pytest.mark.parametrize("tokens", (1, 256, 257, 512, 513))  # both sides of where a token takes more threads
@pytest.mark.parametrize("width", (1024, 1028, 2048, 3072, 4096))
def test_step_of_few_tokens(width, tokens):
    s = 3
    g = torch.Generator(device="cuda").manual_seed(tokens)
    rnd = lambda *sh: torch.randn(*sh, generator=g, device="cuda")  # noqa: E731
    x, y = rnd(tokens, s, width), rnd(tokens, width).bfloat16()
    mix, out, in_, w = rnd(s, s), rnd(s), rnd(s), rnd(width)
    ref = torch.einsum("tfd,fs->tsd", x.double(), mix.double()) + out.double()[:, None] * y.double()[:, None]
    u = torch.einsum("tsd,s->td", ref, in_.double())
    h = u * torch.rsqrt(u.pow(2).mean(1, keepdim=True) + 1e-5) * w.double()
    got = hyper_step(x, y, mix, out, in_, w, 1e-5)
    assert float((x.double() - ref).abs().max()) < 1e-5 * float(ref.abs().max())  # four products and sums in fp32
    assert bool(((got.double() - h).abs() <= 2.0 ** -8 * h.abs() + 1e-4).all())


def _step(m, rows, seed=3):
    """Inputs of a decode step of ``rows`` sequences, and of one prompt of as many tokens."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    i32 = dict(dtype=torch.int32, device="cuda")
    ctx = torch.randint(1, 300, (rows,), generator=g, **i32)
    tables = torch.stack([torch.randperm(127, generator=g, device="cuda")[:16].int() + 1 for _ in range(rows)])
    tokens, slots = torch.randint(0, 512, (128,), generator=g, **i32), torch.full((rows,), -1, **i32)
    pos = torch.arange(128, **i32)
    return (tokens[:rows], ctx - 1, slots, tables, ctx), (tokens, pos, torch.where(pos < rows, pos + 32, -1).int(), [0], [rows], [128])


@pytest.mark.parametrize("rows", (1, 8, 9, 16, 17, 32, 33, 48, 49, 64, 96))
@pytest.mark.parametrize("hidden,heads", ((2048, 16), (1024, 8)))  # layers in slices from 33 rows on, and without them
def test_small_steps_repeat_and_agree_with_the_unfused_layers(hidden, heads, rows):
    from kgs.models.llama import LlamaConfig
    from kgs.serve.model import ServingModel

    c = LlamaConfig(hidden=hidden, layers=2, heads=heads, kv_heads=heads // 4, intermediate=12288 if hidden == 2048 else 1024, vocab=512)
    m = ServingModel(c, device="cuda", num_pages=128, max_model_len=1024)
    m.cache.data.normal_(generator=torch.Generator(device="cuda").manual_seed(rows))
    decode, prompt = _step(m, rows)

    def both():
        m.cache.data[:, 1:32].zero_()
        return m.prefill(*prompt).float(), m.decode(*decode).float(), m.cache.data.float()

    got = both()
    for _ in range(2):
        assert all(torch.equal(a, b) for a, b in zip(got, both()))
    m.fused_max_batch = 0
    for a, b in zip(got, both()):
        assert float((a - b).norm() / b.norm()) < 2e-2  # sums in another order, rounded to bf16 through two layers


# slices of twice the K that one workgroup a CU would have
@pytest.mark.parametrize("m,n,k", ((1, 4096, 2048), (16, 4096, 4096), (48, 4096, 8192), (96, 4096, 2048), (128, 4096, 4096), (33, 2048, 2048), (97, 2048, 1024)))
def test_longer_slices_sum_their_halves_apart(m, n, k):
    from kgs.ops import _lib

    x, w = _operands(m, n, k, 5)
    rule, slabs = (D.slab_split, D.skinny_slabs) if m <= 96 else (D.wide_split, D.wide_slabs)
    assert rule(m, n, k) == (1, 4)
    pw, p = D.PackedWeight(w), torch.empty(8, m, n, device="cuda")
    rc = _lib.lib().kgs_wide_slabs(pw.data.data_ptr(), x.data_ptr(), p.data_ptr(), m, n, k, x.stride(0), 2 if n >= 4096 else 1, 8, _lib.stream_handle(x.device))
    assert rc == 0 and torch.equal(slabs(x, pw), p[0::2] + p[1::2])  # as many slices' sums, added in pairs


# and of four times: (2048 columns of x, 1024 rows of W) 4 for 16
@pytest.mark.parametrize("m,n,k,most", ((64, 4096, 4096, 8), (64, 2048, 2048, 8), (64, 1024, 2048, 16)))
def test_fewer_slices_lose_no_precision(m, n, k, most):
    """The sums of four slices against 64 bits are no further off than those of the most: the same chains or half as many, then fewer additions."""
    from kgs.ops import _lib

    x, w = _operands(m, n, k, 6)
    pw, p = D.PackedWeight(w), torch.empty(most, m, n, device="cuda")
    assert _lib.lib().kgs_skinny_slabs(pw.data.data_ptr(), x.data_ptr(), p.data_ptr(), m, n, k, x.stride(0), 2 if n >= 4096 else 1, most, _lib.stream_handle(x.device)) == 0
    ref = x.double() @ w.double().T

    def off(parts):
        total = parts[0]
        for part in parts[1:]:
            total = total + part
        return float((total.double() - ref).pow(2).mean())

    assert off(D.skinny_slabs(x, pw)) <= off(p)
