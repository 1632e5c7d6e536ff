"""Four-wave decode tiles for sizes without measured entries: the rule, and its sums in the
kernels that take the slices."""
from __future__ import annotations

import pytest
import torch

from kgs.ops import decode as D

DEV = "cuda"


def test_rule_is_launchable_over_sizes():
    """Equal slices of whole 128-deep K-tiles, at most a workgroup a CU and at least half of them
    wherever K has slices left; nothing for sizes that were measured one by one."""
    for m in (32, 33, 128, 129, 256, 257):
        for n in (128, 768, 3072, 16384, 22016, 32000, 65536, 200):
            for k in (128, 256, 2048, 4608, 8192, 11008, 100):
                for most in (8, 16):
                    r = D.w4x_rule(m, n, k, most)
                    if not 33 <= m <= 256 or n % 128 or k % 128:
                        assert r is None
                    if r is None:
                        continue
                    bn, ns, bm = r
                    wgs = -(-m // bm) * (n // bn) * ns
                    assert bn == 128 and bm in (128, 256) and ns <= most and k % (128 * ns) == 0 and wgs <= D.CUS
                    assert 2 * wgs >= D.CUS or ns == most or k // ns < 512
                    assert ns * m * n <= D.SPLITK_WS_FLOATS
    for _, n, k in D.W4X_TUNED:
        assert all(D.w4x_rule(m, n, k) is None for m in (33, 100, 256))


@pytest.mark.parametrize("m,n,k,taken", [(96, 1024, 1024, "general"), (96, 2560, 7168, "general"), (96, 1024, 4096, "library"), (33, 1536, 1536, "library"),
                                         (100, 32000, 2048, "tiles"), (100, 16384, 4096, "general"), (100, 6144, 4096, "tiles")])
def test_decode_products_that_nothing_sums_are_not_sliced(m, n, k, taken, monkeypatch):
    """Slices by rule are for consumers that take their sums: a launch of its own for it costs more than they give
    (entries measured one by one keep theirs)."""
    import kgs.ops
    from kgs.ops import gemm
    from kgs.serve.model import ServingModel

    calls = []
    monkeypatch.setattr(gemm, "gemm_nt_w4x", lambda *a, nslice=1, **kw: calls.append(("tiles", nslice)))
    monkeypatch.setattr(kgs.ops, "gemm_nt", lambda *a, **kw: calls.append(("general", 1)))
    monkeypatch.setattr(torch, "matmul", lambda *a: calls.append(("library", 1)))

    class M:
        backend, packed, decode_fp8 = "kgs", None, False
        w = [{"o": torch.empty(n, k, dtype=torch.bfloat16, device="meta")}]

    ServingModel._proj(M, torch.empty(m, k, dtype=torch.bfloat16, device="meta"), 0, "o", True)
    assert [c[0] for c in calls] == [taken]
    assert calls[0][1] == 1 or (n, k) in D._MEASURED


@pytest.mark.parametrize("m,n,k,tiles", [(128, 4096, 8192, (8, 128)), (129, 4096, 8192, None), (192, 7168, 5120, None), (256, 5120, 8192, None),
                                         (129, 11008, 8192, None), (129, 16384, 8192, (2, 256)), (256, 14336, 5120, (2, 256)),
                                         (256, 14336, 5248, None), (129, 8192, 4096, (2, 128)), (256, 32768, 8192, (1, 256))])
def test_projections_of_a_long_sum_above_128_rows(m, n, k, tiles, monkeypatch):
    """There the rule's 128-row tiles take up to 48 % more than the general kernel or two slices
    of 256-row ones."""
    from kgs.ops import gemm
    from kgs.ops.linear import Projection

    calls = []
    monkeypatch.setattr(gemm, "gemm_nt_w4x", lambda *a, nslice, bm, **kw: calls.append((nslice, bm)) or a[0])
    monkeypatch.setattr(gemm, "gemm_nt", lambda *a, **kw: calls.append(None) or a[0])
    p = Projection(torch.empty(n, k, dtype=torch.bfloat16, device="meta"))
    p._plain(torch.empty(m, k, dtype=torch.bfloat16, device="meta"), m, n, k)
    assert calls == [tiles]


@pytest.mark.gpu
@pytest.mark.parametrize("m", [33, 128, 129, 256])
@pytest.mark.parametrize("n,k", [(128, 128), (768, 2048), (3072, 2048), (2048, 8192), (5120, 1408), (32000, 512), (13056, 4352)])
def test_projection_and_partials(m, n, k):
    """Against the fp64 product: fp32 sums of exact bf16 products in any order (error below
    k 2^-24 of the sum of magnitudes), then one rounding to bf16."""
    from kgs.ops.gemm import gemm_nt_w4x_partials
    from kgs.ops.linear import Projection

    torch.manual_seed(m + n)
    x, w = torch.randn(m, k, device=DEV).bfloat16(), torch.randn(n, k, device=DEV).bfloat16()
    want = x.double() @ w.double().T
    tol = (x.double().abs() @ w.double().abs().T) * k * 2.0 ** -24
    y = Projection(w)(x).double()
    assert bool(((y - want).abs() <= tol + (want.abs() + tol) * 2.0 ** -8).all())
    r = D.w4x_rule(m, n, k)
    if r is not None and r[1] > 1:
        parts = gemm_nt_w4x_partials(x, w, *r, nt_weights=True, private=True)
        assert parts.shape == (r[1], m, n)
        assert bool(((parts.double().sum(0) - want).abs() <= tol).all())


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [2048, 8192])
def test_sixteen_slices_into_norm_and_rotation(cols):
    """The sixteen-slice forms add as the run-time loop does: bits of the sum's own rounding."""
    from kgs.ops.transformer import add_rmsnorm, rope_tables, splitk_add_rmsnorm

    torch.manual_seed(cols)
    rows, ns = 37, 16
    parts = torch.randn(ns, rows, cols, device=DEV)
    d = parts[0].clone()
    for i in range(1, ns):
        d += parts[i]
    x = torch.randn(rows, cols, device=DEV).bfloat16()
    w = torch.randn(cols, device=DEV).bfloat16()
    x1, x2 = x.clone(), x.clone()
    y = splitk_add_rmsnorm(parts, x1, w)
    yw = add_rmsnorm(x2, d.bfloat16(), w)
    assert torch.equal(x1, x2)
    torch.testing.assert_close(y.float(), yw.float(), rtol=2.0 ** -7, atol=1e-6)  # the row sum's order differs: an ulp
    heads, kv = cols // 128 - 8, 4
    cos, sin = rope_tables(64, 128, 1e4, DEV)
    pos, slot = torch.arange(rows, device=DEV, dtype=torch.int32), torch.arange(rows, device=DEV, dtype=torch.int32) + 3
    caches = [torch.zeros(4, kv, 2, 4096, device=DEV, dtype=torch.bfloat16) for _ in range(2)]
    q1, q2 = torch.empty(rows, cols, device=DEV, dtype=torch.bfloat16), d.bfloat16()
    D.rope_cache_(q1, cos, sin, pos, slot, caches[0], heads, kv, partials=parts)
    D.rope_cache_(q2, cos, sin, pos, slot, caches[1], heads, kv)
    assert torch.equal(q1, q2) and torch.equal(*caches)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [1, 681, 682, 683, 700])
def test_rope_forms_by_rows(tokens):
    """Either side of the row count where eight heads share a thread: the same bits as row by row."""
    heads, kv = 16, 4
    torch.manual_seed(tokens)
    qkv = torch.randn(tokens, (heads + 2 * kv) * 128, device=DEV).bfloat16()
    from kgs.ops.transformer import rope_tables

    cos, sin = rope_tables(1024, 128, 1e4, DEV)
    pos = torch.randperm(1024, device=DEV)[:tokens].int()
    slot = torch.randperm(32 * 32, device=DEV)[:tokens].int() - 2
    ca, cb = (torch.zeros(32, kv, 2, 4096, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    one = qkv.clone()
    D.rope_cache_(qkv, cos, sin, pos, slot, ca, heads, kv)
    for a in range(0, tokens, 99):
        D.rope_cache_(one[a:a + 99], cos, sin, pos[a:a + 99].clone(), slot[a:a + 99].clone(), cb, heads, kv)
    assert torch.equal(qkv, one) and torch.equal(ca, cb)
