"""Launches that take single waves as workgroups up to a size (row_waves in transformer.hip, kgs_rope_cache_bf16): both sides of it."""
import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("own_rng")]
DEV = "cuda"


@pytest.mark.parametrize("rows", [1, 5, 1023, 1024, 1025, 1027])
@pytest.mark.parametrize("add", [False, True])
def test_norm_rows(rows, add):
    from kgs.ops.transformer import add_rmsnorm

    x, d, w = (torch.randn(*s, device=DEV).bfloat16() for s in ((rows, 512), (rows, 512), (512,)))
    want = (x.float() + d.float()).bfloat16() if add else x.clone()
    guard = torch.full((rows + 1, 512), 7.0, device=DEV).bfloat16()
    add_rmsnorm(x, d if add else None, w, out=guard[:rows])
    f = want.double()
    ref = f * torch.rsqrt(f.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()
    assert torch.equal(x, want) and bool((guard[rows] == 7).all())
    # one rounding to bf16 and a few of fp32
    assert float(((guard[:rows].double() - ref).abs() - 2.0 ** -8 * ref.abs()).max()) <= 1e-6


@pytest.mark.parametrize("tokens,heads,kv,slices", [(1, 2, 1, 0), (33, 2, 1, 2), (2048, 2, 1, 0), (2049, 2, 1, 0), (2048, 2, 1, 8),
                                                    (2049, 2, 1, 8), (1023, 4, 2, 0), (1024, 4, 2, 0), (2048, 4, 2, 4),
                                                    (768, 2, 1, 2), (769, 2, 1, 2)])
def test_rotation_and_cache(tokens, heads, kv, slices):
    from kgs.ops import decode as D

    nh = heads + 2 * kv
    cos, sin = (torch.randn(300, 64, device=DEV) for _ in range(2))
    pos = torch.randint(0, 300, (tokens,), device=DEV, dtype=torch.int32)
    slot = torch.randperm((tokens // 32 + 2) * 32, device=DEV)[:tokens].int()
    slot[::7] = -1
    cache = torch.zeros(tokens // 32 + 2, kv, 2, 4096, device=DEV).bfloat16()
    part = torch.randn(max(1, slices), tokens, nh * 128, device=DEV)
    total = part[0]
    for p in part[1:]:
        total = total + p
    qkv = torch.full((tokens + 1, nh * 128), 7.0, device=DEV).bfloat16()
    given = total.bfloat16()
    if not slices:
        qkv[:tokens] = given
    D.rope_cache_(qkv[:tokens], cos, sin, pos, slot, cache, heads, kv, partials=part if slices else None)
    rot = D.ref_rope_rows(given, cos, sin, pos, heads + kv).double()
    got = qkv[:tokens].double()
    n = (heads + kv) * 128
    assert float(((got[:, :n] - rot).abs() - 2.0 ** -8 * rot.abs()).max()) <= 1e-5  # fp32 turned, one rounding
    assert torch.equal(qkv[:tokens, n:], given[:, n:]) and bool((qkv[tokens] == 7).all())
    ref = torch.zeros_like(cache)
    k, v = (qkv[:tokens, a:a + kv * 128].reshape(tokens, kv, 128) for a in (heads * 128, n))
    D.ref_cache_write(ref, k, v, slot)
    assert torch.equal(cache, ref)


@pytest.mark.parametrize("M,N,K", [(1, 256, 64), (64, 200, 128), (65, 128, 128), (33, 72, 200), (64, 136, 328), (17, 64, 1024),
                                   (1, 4033, 64), (64, 4040, 320), (33, 4104, 1024), (17, 4032, 128), (65, 4104, 128), (48, 4104, 72)])
def test_small_tiles_by_either_cache_policy(M, N, K):
    """One row tile with whole-line rows of a B of 64 column tiles (non-temporal); fewer of them, two row tiles, rows off the lines."""
    from kgs.ops import _lib

    a, b = (torch.randn(r, K, device=DEV).bfloat16() for r in (M, N))
    c = torch.full((M + 1, N), 7.0, device=DEV).bfloat16()
    rc = _lib.lib().kgs_gemm_bf16_nt_any(a.data_ptr(), b.data_ptr(), c.data_ptr(), None, M, N, K, K, K, N, 0, 64, 64, 1, None,
                                         _lib.stream_handle(a.device))
    want = a.double() @ b.double().T
    assert rc == 0 and bool((c[M] == 7).all())
    assert float((c[:M].double() - want).norm() / want.norm()) < 2.0 ** -8  # one rounding to bf16


@pytest.mark.parametrize("m", [17, 31, 32])
@pytest.mark.parametrize("n,k", [(6272, 2048), (8064, 1024), (8192, 2048)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_skinny_products_in_one_round_of_two_tile_workgroups(m, n, k, swiglu):
    """bf16 outputs of fp32 sums over K: 2^-8 of the largest (a rounding is 2^-9, a fused gate's are two)."""
    from kgs.ops import decode as D

    g = torch.Generator(device="cuda").manual_seed(n + m)
    w = (torch.randn(n, k, device="cuda", generator=g) * k ** -0.5).bfloat16()
    x = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    assert D.skinny_rule(m, n, k) == (23, 1)
    # weights packed with RoPE: one tile a wave, a second round of workgroups
    assert D.skinny_rule(m, n, k, one=True) == ((22, 1) if m * k <= 48 << 10 else (5, 2))
    got = D.skinny_gemm(x, D.PackedWeight(w, swiglu=swiglu)).double()
    want = x.double() @ w.double().T
    if swiglu:
        want = torch.nn.functional.silu(want[:, :n // 2]) * want[:, n // 2:]
    assert (got - want).abs().max() < 2.0 ** -8 * want.abs().max()
