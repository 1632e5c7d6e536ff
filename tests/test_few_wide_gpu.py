"""Products of 17 to 32 rows with x by LDS (native/kernels/decode_few.hip), each of its splits: one tile a workgroup, two on eight waves, two on four;
K of one ring round and of several."""
import pytest
import torch

from kgs.ops import decode as D

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("own_rng")]

SHAPES = ((16, 1024), (4096, 1024), (2048, 8192), (4128, 1024), (8192, 2048), (8224, 1024), (16384, 2048))


def _close(got, ref, factors=1):
    """One rounding to bf16 (2^-9 of the value) and fp32 sums of at most 8192 products (1e-5 of the rows' size) for each factor."""
    err = (got.double() - ref).abs()
    assert bool((err <= 2.0 ** -8 * ref.abs() + 2e-5 * factors * ref.abs().max()).all()), err.max()


@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("m", (17, 24, 32))
def test_each_epilogue(n, k, m):
    x = torch.randn(m, k + 8, device="cuda").bfloat16()[:, :k]  # rows further apart than they are long
    w = (torch.randn(n, k, device="cuda") * k ** -0.5).bfloat16()
    assert D.few_wide(m, n, k) and not D.few_takes(m, n, k)
    pw, ref = D.PackedWeight(w), x.double() @ w.double().T
    _close(D.skinny_few(x, pw), ref)
    normed = ref * torch.rsqrt(x.double().pow(2).mean(1, keepdim=True) + 1e-3)
    _close(D.skinny_few(x, pw, norm=True, eps=1e-3), normed)
    out = torch.randn(m, n, device="cuda").bfloat16()
    want = out.double() + ref
    assert D.own_gemm(x, pw, out=out, resid=True) is out
    _close(out, want)
    if n % 32 == 0:
        g, u = normed.chunk(2, 1)
        _close(D.skinny_few(x, D.PackedWeight(w, swiglu=True), norm=True, eps=1e-3), torch.nn.functional.silu(g) * u, 4)


@pytest.mark.parametrize("heads,kv", ((4, 2), (32, 8), (48, 16)))
@pytest.mark.parametrize("m", (17, 32))
def test_rotation_and_cache_as_the_separate_launch(heads, kv, m):
    from kgs.ops.transformer import rope_tables

    k = 1024
    x, w = torch.randn(m, k, device="cuda").bfloat16(), (torch.randn((heads + 2 * kv) * 128, k, device="cuda") * k ** -0.5).bfloat16()
    cos, sin = rope_tables(256, 128, 10000.0, "cuda")
    pos, slots = torch.arange(m, dtype=torch.int32, device="cuda") * 13 % 200, torch.randperm(8 * 32, device="cuda")[:m].int()
    slots[m // 2] = -1
    caches = [D.PagedKVCache(1, 8, kv, "cuda") for _ in range(2)]
    got = D.skinny_few(x, D.PackedWeight(w, rope=(heads, kv)), norm=True,
                       rope={"cos": cos, "sin": sin, "positions": pos, "slots": slots, "cache": caches[0].layer(0)})
    want = D.skinny_few(x, D.PackedWeight(w), norm=True)  # the same sums, row by row
    D.rope_cache_(want, cos, sin, pos, slots, caches[1].layer(0), heads, kv)
    assert torch.equal(got, want) and torch.equal(caches[0].data, caches[1].data)


def test_what_goes_elsewhere():
    for m, n, k in ((16, 4096, 4096), (33, 4096, 4096), (24, 4096, 1536), (24, 4096, 14336), (24, 28672, 4096), (24, 4112, 1024)):
        assert not D.few_wide(m, n, k), (m, n, k)


# K's parts are summed apart and added in their order, however few waves take them: eight of up to 4096 rows of W and K of 1024, four of up to 8192 rows, else two. One
# tile a workgroup by one, two and eight waves, two tiles by two; a part of four k-steps and of several rounds, its end at every fourth step of a round
@pytest.mark.parametrize("n,k,parts", ((64, 1024, 8), (2048, 1024, 8), (2048, 3072, 8), (4096, 5120, 8), (4096, 8192, 8), (2048, 512, 4), (2048, 2560, 4), (4160, 1024, 4),
                                       (6144, 1536, 4), (8192, 2048, 4), (8256, 512, 2), (16384, 1536, 2), (28672, 1024, 2)))
@pytest.mark.parametrize("m", (1, 5, 13, 16))
def test_parts_are_summed_apart(n, k, parts, m):
    from kgs.ops import _lib

    x, w = torch.randn(m, k, device="cuda").bfloat16(), (torch.randn(n, k, device="cuda") * k ** -0.5).bfloat16()
    pw, p = D.PackedWeight(w), torch.empty(parts, m, n, device="cuda")
    rc = _lib.lib().kgs_skinny_slabs(pw.data.data_ptr(), x.data_ptr(), p.data_ptr(), m, n, k, k, 2 if n >= 4096 and n % 128 == 0 else 1, parts, _lib.stream_handle(x.device))
    assert rc == 0 and D.few_takes(m, n, k)
    want = p[0]
    for part in p[1:]:
        want = want + part
    assert torch.equal(D.skinny_few(x, pw), want.bfloat16())  # the same products in the same order: the same bits


def test_calls_that_only_the_other_kernel_takes():
    """own_gemm of 17 to 32 rows, as it was before these rows had a kernel of few: rows far apart and an out inside a wider one are computed, a norm with a residual is refused."""
    m, n, k, ld = 17, 2048, 1024, (1 << 25) + 8
    w = (torch.randn(n, k, device="cuda") * k ** -0.5).bfloat16()
    pw, rows = D.PackedWeight(w), torch.randn(m, k, device="cuda").bfloat16()
    far = torch.empty((m - 1) * ld + k, device="cuda", dtype=torch.bfloat16).as_strided((m, k), (ld, 1))
    far.copy_(rows)
    ref = rows.double() @ w.double().T
    _close(D.own_gemm(far, pw), ref)
    out = torch.full((m + 2, n), 7.0, device="cuda", dtype=torch.bfloat16)
    D.own_gemm(rows, pw, out=out)
    _close(out[:m], ref)
    assert bool((out[m:] == 7).all())
    with pytest.raises(ValueError):
        D.own_gemm(rows, pw, out=out[:m], norm=True, resid=True)
