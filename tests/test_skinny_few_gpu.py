"""Products of few rows (native/kernels/decode_few.hip) against the plain product in float64: the edges of its splits over waves
and tiles, each epilogue, and the RMSNorm whose statistics it makes itself -- as decode.hip's skinny does up to 64 rows."""
import pytest
import torch

from kgs.ops import decode as D

pytestmark = pytest.mark.gpu

# one strip; one and two rounds of strips with 8, 4 and 2 waves, each side of where the split changes; K at the ring's least
SHAPES = [(16, 512), (4096, 1024), (4096, 1536), (4112, 1024), (8192, 512), (8208, 512), (8192, 4096), (2048, 8192)]


def _operands(m, n, k, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(m, k + 8, generator=g, device="cuda").bfloat16()[:, :k]  # rows further apart than they are long
    return x, (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).bfloat16()


def _close(got, ref, rows_scale=1.0):
    """One rounding to bf16 (2^-9 of the value) and fp32 sums of at most 8192 products (1e-5 of the rows' size)."""
    err = (got.double() - ref).abs()
    assert bool((err <= 2.0 ** -8 * ref.abs() + 2e-5 * ref.abs().max() * rows_scale).all()), err.max()


@pytest.mark.parametrize("m", (1, 5, 16))
@pytest.mark.parametrize("n,k", SHAPES)
def test_product_norm_and_residual(n, k, m):
    x, w = _operands(m, n, k)
    assert D.few_takes(m, n, k)
    pw = D.PackedWeight(w)
    ref = x.double() @ w.double().T
    _close(D.skinny_few(x, pw), ref)
    scale = torch.rsqrt(x.double().pow(2).mean(1, keepdim=True) + 1e-3)
    _close(D.skinny_few(x, pw, norm=True, eps=1e-3), ref * scale)
    out = torch.randn(m, n, device="cuda").bfloat16()
    want = out.double() + ref
    assert D.skinny_few(x, pw, out=out, resid=True) is out
    _close(out, want)


@pytest.mark.parametrize("act", ("silu", "gelu_tanh"))
@pytest.mark.parametrize("n,k,m", ((32, 512, 1), (4128, 1024, 7), (16384, 512, 16)))
def test_gated(n, k, m, act):
    x, w = _operands(m, n, k, 1)
    got = D.skinny_few(x, D.PackedWeight(w, swiglu=True, act=act), norm=True)
    z = x.double() @ w.double().T * torch.rsqrt(x.double().pow(2).mean(1, keepdim=True) + 1e-5)
    g, u = z.chunk(2, 1)
    g = torch.nn.functional.silu(g) if act == "silu" else torch.nn.functional.gelu(g, approximate="tanh")
    _close(got, g * u, rows_scale=4.0)  # both factors' errors


@pytest.mark.parametrize("m", (1, 6, 16))
@pytest.mark.parametrize("heads,kv", ((4, 2), (32, 8), (32, 16)))
def test_rope_and_cache_as_the_separate_launch(heads, kv, m):
    k = 1024
    x, w = _operands(m, (heads + 2 * kv) * 128, k, 2)
    from kgs.ops.transformer import rope_tables

    cos, sin = rope_tables(256, 128, 10000.0, "cuda")
    pos = torch.arange(m, dtype=torch.int32, device="cuda") * 13 % 200
    slots = torch.randperm(8 * 32, device="cuda")[:m].int()
    slots[m // 2] = -1
    caches = [D.PagedKVCache(1, 8, kv, "cuda") for _ in range(2)]
    got = D.skinny_few(x, D.PackedWeight(w, rope=(heads, kv)), norm=True,
                       rope={"cos": cos, "sin": sin, "positions": pos, "slots": slots, "cache": caches[0].layer(0)})
    want = D.skinny_few(x, D.PackedWeight(w), norm=True)  # the same sums, row by row
    D.rope_cache_(want, cos, sin, pos, slots, caches[1].layer(0), heads, kv)
    assert torch.equal(got, want) and torch.equal(caches[0].data, caches[1].data)


# 2, 4 and 8 waves, rings of 1 to 4 k-steps, one and several rounds of them
@pytest.mark.parametrize("n,k", ((16, 64), (48, 192), (2048, 128), (64, 384), (32, 768), (832, 1280), (2048, 768), (16, 2048), (64, 1536)))
@pytest.mark.parametrize("m", (1, 16, 17, 32))
def test_plain_products_of_any_short_sum(n, k, m):
    x, w = _operands(m, n, k, 7)
    pw = D.PackedWeight(w)
    assert D.few_takes(m, n, k, plain=True)
    ref = x.double() @ w.double().T
    _close(D.skinny_few(x, pw), ref)
    out = torch.randn(m, n, device="cuda").bfloat16()
    want = out.double() + ref
    _close(D.skinny_few(x, pw, out=out, resid=True), want)
    if n % 32 == 0:
        g, u = ref.chunk(2, 1)
        _close(D.skinny_few(x, D.PackedWeight(w, swiglu=True)), torch.nn.functional.silu(g) * u, 4.0)


def test_what_it_does_not_take():
    for m, n, k in ((17, 4096, 4096), (0, 4096, 4096), (4, 4096, 768), (4, 4104, 512)):
        assert not D.few_takes(m, n, k)
    for m, n, k in ((33, 4096, 4096), (4, 4096, 96), (4, 4104, 512)):
        assert not D.few_takes(m, n, k, plain=True)
    assert not D.few_takes(4, 4096, 4096, fp8=True)
    x, w = _operands(4, 32, 512)
    with pytest.raises(ValueError):
        D.skinny_few(x, D.PackedWeight(w), resid=True)


def test_infinite_and_missing_values_stay_in_their_rows():
    x, w = _operands(5, 64, 512, 3)
    x = x.clone()
    x[2, 7], x[4, 9] = float("nan"), float("inf")
    got = D.skinny_few(x, D.PackedWeight(w), norm=True).float()
    assert got[2].isnan().all() and got[[0, 1, 3]].isfinite().all() and not (got[4].abs() > 0).logical_and(got[4].isfinite()).any()


# x through LDS in one K slice and in several, K split inside the workgroup, in one and in two tiles; each column tile's edge
@pytest.mark.parametrize("variant,ksplit,n,k,m", [(None, None, *nk, m) for nk in ((6144, 4096), (2048, 2048)) for m in (12, 17, 32, 33, 64)] + [
    (1, 1, 256, 1024, 12), (3, 2, 256, 2048, 16), (4, 4, 128, 2048, 17), (22, 1, 64, 1024, 32), (23, 1, 64, 2048, 31), (10, 2, 192, 1024, 33),
    (24, 1, 64, 1024, 64), (25, 1, 128, 1024, 49)])
def test_skinny_norm_by_its_own_statistics(variant, ksplit, n, k, m):
    x, w = _operands(m, n, k, 4)
    pw = D.PackedWeight(w)
    ref = x.double() @ w.double().T
    want = ref * torch.rsqrt(x.double().pow(2).mean(1, keepdim=True) + 1e-3)
    for _ in range(2):  # the second call finds the first one's slabs and tickets
        got = D.own_gemm(x, pw, norm=True, eps=1e-3) if variant is None else D.skinny_gemm(x, pw, ksplit=ksplit, variant=variant, norm=True, eps=1e-3)
        _close(got, want)
    out = torch.randn(m, n, device="cuda").bfloat16()
    want = out.double() + ref
    _close(D.own_gemm(x, pw, out=out, resid=True), want)


# few rows by 2, 4 and 8 waves; skinny with x through LDS, in K slices, and with K split inside the workgroup
@pytest.mark.parametrize("form,n,k,m", [("few", 8208, 4096, 16), ("few", 4112, 4096, 16), ("few", 4096, 4096, 9), ((1, 1), 256, 4096, 16), ((4, 1), 64, 8192, 32),
                                        ((3, 2), 256, 4096, 16), ((10, 4), 192, 4096, 64), ((22, 1), 64, 4096, 32), ((23, 1), 64, 8192, 31), ((24, 1), 64, 4096, 64)])
@pytest.mark.parametrize("large", (1, 30))
def test_own_statistics_are_sums_rounded_once(form, n, k, m, large):
    """A negative eps close to the mean square lays the sum's last bits open: 1 / scale^2 = ss / k + eps, k a power of two, without a further rounding."""
    g = torch.Generator(device="cuda").manual_seed(k + m)
    v = torch.randn(k, generator=g, device="cuda")
    v[:4] *= large
    v = v.bfloat16()
    x = torch.stack([v[torch.randperm(k, generator=g, device="cuda")] for _ in range(m)])
    w = (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).bfloat16()
    ss = float(v.double().pow(2).sum())
    eps = float(torch.tensor(-ss / k * (1 - 2.0 ** -18), dtype=torch.float32))
    pw = D.PackedWeight(w)
    got = D.skinny_few(x, pw, norm=True, eps=eps) if form == "few" else D.skinny_gemm(x, pw, variant=form[0], ksplit=form[1], norm=True, eps=eps)
    ref = x.double() @ w.double().T
    scale = (got.double() * ref).sum(1) / ref.pow(2).sum(1)  # the rows' outputs differ by their roundings alone
    err = (k * (scale.pow(-2) - eps) / ss - 1).abs()
    # a rounding to fp32 (2^-24), the parts' before they meet in fp64 (a lane's eight values, 3 2^-24 of them; four values of 30 times the others' size are
    # most of the sum), and what 64 roundings to bf16 and more leave of 2^-9 times 2^-18
    assert float(err.max()) <= (1.25 if large == 1 else 3.0) * 2.0 ** -24, float(err.max()) * 2 ** 24


@pytest.mark.parametrize("m", (9, 24, 40))
def test_skinny_rope_by_its_own_statistics(m):
    from kgs.ops.transformer import rope_tables

    for n, k, heads, kv in ((6144, 4096, 32, 8), (3072, 2048, 16, 4)):
        x, w = _operands(m, n, k, 5)
        cos, sin = rope_tables(256, 128, 10000.0, "cuda")
        pos, slots = torch.arange(m, dtype=torch.int32, device="cuda"), torch.randperm(256, device="cuda")[:m].int()
        caches = [D.PagedKVCache(1, 8, kv, "cuda") for _ in range(2)]
        rope = {"cos": cos, "sin": sin, "positions": pos, "slots": slots}
        pw = D.PackedWeight(w, rope=(heads, kv))
        ss = x.float().pow(2).sum(1)
        got = D.own_gemm(x, pw, norm=True, rope={**rope, "cache": caches[0].layer(0)})
        want = D.skinny_gemm(x, pw, rms=ss, rope={**rope, "cache": caches[1].layer(0)})
        # the statistics' last bits and, up to 16 rows, the order of the sums: one unit of bf16 before the rotation
        assert float((got.float() - want.float()).norm() / want.float().norm()) < 2.0 ** -8
        assert float((caches[0].data.float() - caches[1].data.float()).norm() / caches[1].data.float().norm()) < 2.0 ** -8


def test_norm_and_resid_are_refused_where_they_do_not_go():
    x, w = _operands(70, 4096, 2048, 6)
    pw = D.PackedWeight(w)
    ss = torch.zeros(70, device="cuda")
    for kw in ({"norm": True}, {"norm": True, "rms": ss}, {"resid": True}, {"resid": True, "resid_ss": ss, "out": x}):
        with pytest.raises(ValueError):
            D.skinny_gemm(x, pw, **kw)
    assert not D.own_takes(65, 4096, 2048) and not D.own_takes(16, 4096, 2048, fp8=True)


@pytest.mark.parametrize("n,k,gated", ((2048, 768, False), (832, 2048, False), (2048, 128, False), (1504, 2048, False), (16384, 2048, True), (24576, 1024, True),
                                       (32000, 512, False), (96, 64, True)))
@pytest.mark.parametrize("m", (1, 9, 16, 17, 32, 33, 64, 96, 97))
def test_projections_by_the_packed_weight(n, k, gated, m):
    from kgs.ops.linear import Projection

    x, w = _operands(m, n, k, 8)
    ref = x.double() @ w.double().T
    if gated:
        g, u = ref.chunk(2, 1)
        ref = torch.nn.functional.silu(g) * u
    got = Projection(w, "silu" if gated else None)(x)
    assert got.shape == ref.shape
    # some routes round gate and up to bf16 before the product
    assert bool(((got.double() - ref).abs() <= 2.0 ** -7 * ref.abs() + 2.0 ** -7 * (ref.abs().max() if gated else 0) + 1e-4 * ref.abs().max()).all())


@pytest.mark.parametrize("m,n,k", [(1, 16, 64), (16, 2048, 128), (7, 4128, 1024), (24, 2048, 192), (32, 48, 512)])
def test_two_products(m, n, k):
    """One launch's bits are two launches', of operands that are columns of a wider matrix."""
    z, (_, w), (_, w2) = torch.randn(m, 2 * k + 8, device="cuda").bfloat16(), _operands(m, n, k), _operands(m, n, k, 1)
    x, x2, pw, pw2 = z[:, :k], z[:, k + 8:], D.PackedWeight(w), D.PackedWeight(w2)
    got, got2 = D.skinny_few_two(x, pw, x2, pw2)
    assert torch.equal(got, D.skinny_few(x, pw)) and torch.equal(got2, D.skinny_few(x2, pw2))
    with pytest.raises(ValueError):
        D.skinny_few_two(x, pw, torch.empty(m, k, device="cuda", dtype=torch.bfloat16), pw2)


@pytest.mark.parametrize("n,k,gated", ((2048, 768, False), (24576, 512, False), (256, 512, False), (16384, 1024, True)))
@pytest.mark.parametrize("m", (1, 8, 32, 40))
def test_projections_of_rows_that_the_packed_kernels_cannot_read(n, k, gated, m):
    """Columns, odd addresses and, of plain weights, one row repeated or rows that overlap go where any matrix goes, in each of the ways in."""
    from kgs.ops.linear import Projection

    g = torch.Generator(device="cuda").manual_seed(m)
    z, (_, w) = torch.randn(m + 1, k + 8, generator=g, device="cuda").bfloat16(), _operands(m, n, k, 9)
    p, q = Projection(w, "silu" if gated else None), Projection(w, "silu" if gated else None)
    rows = z[:m, :k]
    spread = torch.empty(m, 2 * k, device="cuda", dtype=torch.bfloat16)[:, ::2].copy_(rows)
    over = () if gated else (rows[:1].expand(m, k), z.flatten().as_strided((m, k), (8, 1)))
    for x in (rows.t().contiguous().t(), spread, z[:m, 1:k + 1], *over):
        ref = x.double() @ w.double().T
        if gated:
            a, b = ref.chunk(2, 1)
            ref = torch.nn.functional.silu(a) * b
        for got in (p(x), *p.two(x, q, x), p.partials(x)):
            # one rounding to bf16 and fp32 sums; of a gate with its factors rounded before
            tol = 2.0 ** -7 * ref.abs() + 2.0 ** -7 * (ref.abs().max() if gated else 0) + 1e-4 * ref.abs().max()
            got = got.sum(0) if got.dim() == 3 else got
            assert got.shape == ref.shape and bool(((got.double() - ref).abs() <= tol).all())


@pytest.mark.parametrize("n,k", ((2048, 8192), (2048, 11008), (8192, 8192), (5120, 13824)))  # K in two halves, off 512, and both kernels' sides
@pytest.mark.parametrize("m", (1, 4, 9, 16))
def test_residual_products_of_long_sums(n, k, m):
    x, w = _operands(m, n, k, 10)
    pw = D.PackedWeight(w)
    ref = x.double() @ w.double().T
    for counters in (None, torch.zeros(n // 16, dtype=torch.int32, device="cuda")):
        for _ in range(2):  # the second call finds the first one's slabs and tickets
            out = torch.randn(m, n, device="cuda").bfloat16()
            want = out.double() + ref
            _close(D.own_gemm(x, pw, out=out, resid=True, counters=counters), want)
