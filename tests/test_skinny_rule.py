"""Skinny GEMM variants by rule: launchable over sizes, and the forms with the K split inside the
workgroup for up to 64 rows."""
from __future__ import annotations

from fractions import Fraction

import pytest
import torch

from kgs.ops import decode as D

DEV = "cuda"


def test_rule_is_launchable():
    for m in (1, 16, 17, 32, 33, 40, 48, 64):
        for n in (64, 128, 1280, 2048, 4096, 4160, 6144, 6208, 16384):
            for k in (512, 1024, 1536, 2048, 4096, 5120, 8192, 9216):
                for one in (False, True):
                    v, ks = D.skinny_rule(m, n, k, one)
                    rps, kpc, _ = D.skinny_geometry(m, v)
                    if n % 64 == 0 and k % 512 == 0:  # what callers pack weights of
                        assert n % rps == 0 and k % kpc == 0 and (k // kpc) % ks == 0, (m, n, k, v, ks)
                    assert not one or D.SKINNY_VARIANTS[v][0] == 1 or m > 64


def test_rule_keeps_to_where_its_forms_are_the_faster():
    """Where all of x per workgroup, a second round of workgroups or short slices cost more than they give."""
    kin = set()
    for m in (1, 8, 16, 17, 24, 32, 40, 64):
        for n in (1024, 1280, 2048, 3072, 4096, 5120, 6144, 9216):
            for k in (1024, 2048, 2560, 3072, 4096, 5120, 8192, 10240):
                v, ks = D.skinny_rule(m, n, k)
                strips = n // (16 * D.SKINNY_VARIANTS[v][0])
                if v in D.KIN_VARIANTS:
                    kin.add((m, n, k))
                    assert ks * strips <= 384 and (strips <= 256 or m <= 16 and m * k <= 32 << 10)
                elif m > 16:
                    assert k // ks >= 512 or ks <= D.choose_ksplit(m, n, k)
    assert not kin & {(16, 5120, 3072), (16, 5120, 5120), (16, 3072, 8192), (32, 5120, 3072), (32, 1024, 4096), (40, 5120, 3072), (16, 6144, 4096)}
    assert kin >= {(16, 4096, 4096), (16, 2048, 8192), (8, 6144, 4096), (24, 6144, 2048), (32, 4096, 4096), (40, 6144, 2048), (64, 2048, 2048)}
    assert D.skinny_rule(24, 5120, 10240)[0] == 4 and D.skinny_rule(24, 16384, 2048)[0] == 5 and D.skinny_rule(48, 1024, 4096) == (10, 8)


class _Weight:
    def __init__(self, n, k, rope=None, fp8=False):
        self.n, self.k, self.rope, self.fp8 = n, k, rope, fp8


def test_what_the_skinny_gemm_takes():
    """Its own choice of a variant has to tile the weight, and the rotation's to have one-tile waves."""
    for m in range(1, 258):
        for n, k, fp8, rope in ((3072, 2048, False, False), (3072, 2048, False, True), (3072, 2048, True, False), (3136, 2048, False, False),
                                (2048, 2304, False, False)):
            ok = D.skinny_takes(m, n, k, fp8, rope)
            if m > (64 if rope or fp8 else 256):
                assert not ok
                continue
            v, ks = D._skinny_plan(m, n, k, fp8, rope)
            rps, kpc, _ = D.skinny_geometry(m, v)
            assert ok == (n % rps == 0 and k % kpc == 0) and (not ok or (k // kpc) % ks == 0)
            assert not rope or D.SKINNY_VARIANTS[v][0] == 1
    assert D.skinny_takes(64, 3072, 2048, rope=True) and D.skinny_takes(200, 3072, 2048)
    assert not D.skinny_takes(200, 3136, 2048) and not D.skinny_takes(1, 2048, 2304)


@pytest.mark.parametrize("most,rows,fused", [(48, 48, True), (48, 49, False), (128, 64, True), (128, 65, False), (300, 257, False), (0, 1, False)])
def test_prompt_rows_of_the_fused_layer(most, rows, fused):
    """A larger fused_max_batch takes no prompt to products that are not built for it."""
    from kgs.serve.model import ServingModel

    class M:
        decode_fp8, fused_max_batch = False, most
        packed = [{"qkv": _Weight(3072, 2048, rope=(16, 4)), "o": _Weight(2048, 2048), "gate_up": _Weight(16384, 2048), "down": _Weight(2048, 8192)}]
        packed_lm = _Weight(1024, 2048)

    assert ServingModel._fused_prompts(M, rows, 1) is fused


@pytest.mark.parametrize("most,rows,slabs", [(48, 33, True), (48, 96, True), (48, 97, False), (48, 32, False), (33, 64, True), (32, 33, False), (16, 40, False),
                                             (16, 96, False), (0, 64, False)])
def test_rows_of_the_layers_in_slices(most, rows, slabs):
    """fused_max_batch bounds these layers too: where the caller wants few rows on packed weights, larger steps take the split tiles."""
    from types import SimpleNamespace

    from kgs.serve.model import ServingModel

    class M:
        decode_fp8, backend, fuse_splitk, rope_attn, fused_max_batch = False, "kgs", True, False, most
        packed = [{"qkv": _Weight(3072, 2048, rope=(16, 4)), "o": _Weight(2048, 2048), "gate_up": _Weight(16384, 2048), "down": _Weight(2048, 8192)}]
        packed_lm, cfg = _Weight(1024, 2048), SimpleNamespace(hidden=2048)

    assert ServingModel._slabs(M, rows) is slabs
    M._slabs = staticmethod(lambda m: ServingModel._slabs(M, m))
    assert ServingModel._slabs_pay(M, rows) is slabs
    M.packed = [{**M.packed[0], "down": _Weight(2048, 11008)}]  # slices badly: from 49 rows on the split tiles are the faster
    assert ServingModel._slabs_pay(M, rows) is (slabs and rows <= 48)


def test_what_tiles_for_prompts_makes_its_own_statistics():
    for n in (64, 128, 1024, 1280, 2048, 3072, 4096, 6144, 8192, 10240, 28672, 32000, 128256, 262144):
        for k in (512, 1024, 1536, 2048, 2560, 4096, 5120, 8192, 9216, 12288):
            for m in (1, 2, 8, 9, 16, 17, 24, 32, 33, 48, 64):
                for rope in (False, True):
                    assert D.own_takes(m, n, k, False, rope) or not D.skinny_takes(m, n, k, False, rope), (m, n, k, rope)


def test_what_the_rules_of_slices_take_the_kernel_takes():
    """Addresses off 16 bytes are refused after the sizes and before any launch, so the entries tell here whether they take the sizes."""
    from kgs.ops import _lib

    lib = _lib.lib()
    align = lib.kgs_skinny_slabs(1, 1, 1, 1, 64, 128, 128, 1, 1, None)
    assert align not in (0, lib.kgs_skinny_slabs(1, 1, 1, 97, 64, 128, 128, 1, 1, None))
    for n in (64, 128, 192, 2048, 4096, 4160, 28672, 128256, 256000, 262208, 1 << 20):
        for k in (128, 256, 384, 2048, 4096, 8192, 12288, 14336, 16384, 65536):
            for m in (1, 16, 17, 32, 33, 64, 65, 96):
                split, tiles = D.slab_split(m, n, k), D.slab_rows_tiles(m, n, k)
                if split:
                    assert lib.kgs_skinny_slabs(1, 1, 1, m, n, k, k, *split, None) == align, (m, n, k)
                if tiles:
                    assert lib.kgs_skinny_rows(1, 1, 1, m, n, k, k, n, tiles, 0, None, 0.0, 0.0, None) == align, (m, n, k)


def test_what_the_rules_of_wide_slices_take_the_kernel_takes():
    from kgs.ops import _lib

    lib = _lib.lib()
    align = lib.kgs_wide_slabs(1, 1, 1, 128, 64, 128, 128, 1, 1, None)
    assert align not in (0, lib.kgs_wide_slabs(1, 1, 1, 129, 64, 128, 128, 1, 1, None))
    for n in (64, 192, 2048, 4096, 4160, 28672, 128256, 1 << 20):
        for k in (128, 384, 2048, 11008, 65536):
            for m in (96, 97, 128, 129):
                split, head = D.wide_split(m, n, k), D.head_pays(m, n, k)
                assert (split is None) is (m not in (97, 128) or n % 64 != 0)
                if split:
                    assert lib.kgs_wide_slabs(1, 1, 1, m, n, k, k, *split, None) == align, (m, n, k)
                if head:
                    assert lib.kgs_wide_rows(1, 1, 1, m, n, k, k, n, D._rows_tiles(m, n, k, D.CUS), None, 0.0, None) == align, (m, n, k)
    for m, n, k, pays in ((48, 32000, 4096, False), (49, 32000, 4096, True), (128, 32000, 2048, True), (64, 32000, 1024, False), (64, 128256, 4096, False),
                          (100, 40960, 4096, False), (128, 64000, 4096, True), (129, 32000, 4096, False)):
        assert D.head_pays(m, n, k) is pays, (m, n, k)


def test_few_rows_keep_to_where_they_are_the_faster():
    """Beside skinny: not for wide weights of short sums, x that is long, strips at multiples of 256 KB; beside the library: neither long sums nor wide weights."""
    few = [(1, 28672, 4096), (8, 32000, 4096), (8, 16384, 2048), (1, 24576, 2048), (8, 10240, 1024), (16, 6144, 4096), (8, 4096, 14336), (1, 4096, 4096), (16, 2048, 3584),
           (4, 8192, 8192), (24, 2048, 768), (24, 4096, 1536), (32, 832, 1984), (8, 22016, 768), (12, 2048, 11008)]
    not_few = [(1, 64000, 1024), (8, 64000, 2048), (1, 32000, 2048), (8, 32000, 5120), (4, 24576, 512), (1, 4096, 8192), (8, 8192, 8192), (16, 8192, 8192), (8, 1024, 14336),
               (16, 2048, 8192), (12, 1024, 6144), (24, 2048, 1024), (32, 4096, 1024), (24, 896, 4864), (32, 2048, 11008), (16, 13824, 768), (16, 6144, 11008), (4, 5120, 13824)]
    for case in few:
        assert D.few_route(*case, True), case
    for case in not_few:
        assert not D.few_route(*case, True), case


def test_whole_products_keep_to_where_they_are_the_faster():
    for m, n, k, gated, pay in ((24, 16384, 2048, True, True), (32, 10240, 2048, True, True), (32, 10240, 8192, True, False), (24, 4096, 4096, True, False), (32, 8192, 14336, True, False),
                                (24, 16384, 768, True, False), (24, 16384, 2048, False, False), (16, 16384, 2048, True, False), (64, 28672, 4096, True, True), (90, 28672, 5120, True, True),
                                (64, 32000, 1024, True, False), (96, 24576, 2048, True, False), (64, 32000, 4096, False, True), (96, 32000, 4096, False, True), (64, 24576, 512, False, False),
                                (64, 40960, 4096, False, False), (64, 64000, 4096, False, True), (64, 32000, 2048, False, False), (96, 64000, 2048, False, False), (96, 128256, 4096, False, False), (97, 32000, 4096, False, False)):
        assert D.rows_pay(m, n, k, gated) is pay, (m, n, k, gated)


def test_slices_keep_to_where_they_are_the_faster():
    for m, n, k, fill in ((64, 4096, 11008, False), (49, 2048, 11008, False), (96, 2560, 14336, False), (64, 512, 5632, False), (96, 4096, 14336, True), (96, 2048, 5632, True),
                          (64, 8192, 28672, True), (64, 2048, 8192, True), (64, 2080, 2048, False)):
        assert D.slabs_fill(m, n, k) is fill, (m, n, k)
    for m, n, k, pay in ((1, 2048, 2048, True), (1, 4096, 4096, False), (8, 4096, 4096, False), (16, 4096, 4096, False), (24, 4096, 4096, True), (32, 4096, 1024, False),
                         (32, 2048, 8192, True), (1, 1024, 13824, False), (32, 4096, 11008, False), (64, 4096, 11008, False), (64, 2048, 8192, True), (96, 4096, 1024, False),
                         (8, 4096, 14336, True), (97, 2048, 2048, False)):
        assert D.slabs_pay(m, n, k) is pay, (m, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("m,v", [(17, 22), (32, 22), (24, 23), (33, 24), (64, 24), (40, 25)])
def test_k_split_in_the_workgroup(m, v):
    """Against fp32 for every epilogue: plain, split, RMS + SwiGLU, residual with its sums of squares, and
    (one-tile waves) RoPE with the cache write, whose bits are the plain output's through rope_cache_."""
    from kgs.ops.transformer import rope_tables

    torch.manual_seed(m)
    n, k = 512, 2048
    x = torch.randn(m, k, device=DEV).bfloat16()
    w = (torch.randn(n, k, device=DEV) * k ** -0.5).bfloat16()
    ref = x.float() @ w.float().T
    # fp32 sums of k exact products (k 2^-24 of their magnitudes) and one rounding to bf16
    tol = k * 2.0 ** -24 * (x.float().abs() @ w.float().abs().T) + 2.0 ** -8 * ref.abs()
    pw = D.PackedWeight(w)
    for ks in (1, 2):
        y = D.skinny_gemm(x, pw, variant=v, ksplit=ks).float()
        assert bool(((y - ref).abs() <= tol).all())
        res = torch.randn(m, n, device=DEV).bfloat16()
        old, ss = res.float(), torch.zeros(m, device=DEV)
        D.skinny_gemm(x, pw, out=res, resid_ss=ss, variant=v, ksplit=ks)
        assert bool(((res.float() - old - ref).abs() <= tol + 2.0 ** -8 * (old + ref).abs()).all())
        torch.testing.assert_close(ss, res.float().pow(2).sum(-1), rtol=1e-4, atol=1e-3)
    ss = x.float().pow(2).sum(-1).contiguous()
    wide = (torch.randn(2 * n, k, device=DEV) * k ** -0.5).bfloat16()
    xn = x.float() * torch.rsqrt(ss / k + 1e-5)[:, None]
    g, u = xn @ wide[:n].float().T, xn @ wide[n:].float().T
    got = D.skinny_gemm(x, D.PackedWeight(wide, swiglu=True, fold=torch.ones(k, device=DEV)), rms=ss, variant=v, ksplit=1)
    torch.testing.assert_close(got.float(), torch.nn.functional.silu(g) * u, rtol=2e-2, atol=1e-3)
    if D.SKINNY_VARIANTS[v][0] != 1:
        return
    heads, kv = 4, 2
    wq = (torch.randn((heads + 2 * kv) * 128, k, device=DEV) * k ** -0.5).bfloat16()
    one = torch.ones(k, device=DEV)
    cos, sin = rope_tables(256, 128, 1e4, DEV)
    pos, slot = torch.arange(m, device=DEV, dtype=torch.int32) * 3, torch.arange(m, device=DEV, dtype=torch.int32) - 1
    ca, cb = (torch.zeros(4, kv, 2, 4096, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    q1 = D.skinny_gemm(x, D.PackedWeight(wq, fold=one), rms=ss, variant=v, ksplit=1)
    D.rope_cache_(q1, cos, sin, pos, slot, ca, heads, kv)
    q2 = D.skinny_gemm(x, D.PackedWeight(wq, fold=one, rope=(heads, kv)), rms=ss, variant=v, ksplit=1,
                       rope={"cos": cos, "sin": sin, "positions": pos, "slots": slot, "cache": cb})
    assert torch.equal(q1, q2) and torch.equal(ca, cb)


def _exact(words) -> float:
    """An exact sum's value from its eight integers (decode.hip add_exact), rounded once."""
    w = [int(x) & (2 ** 64 - 1) for x in words]
    if w[-1] >> 62:
        return float("nan") if w[-1] >> 62 & 1 else float("inf")
    return float(Fraction(sum(x << 32 * i for i, x in enumerate(w)), 2 ** 149))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1024, 8192])
@pytest.mark.parametrize("m,variant,ksplit", [(8, 1, 1), (8, 1, 4), (8, 20, 1), (24, 22, 1), (24, 5, 2), (48, 24, 1), (64, 10, 4), (64, 25, 1), (64, 12, 1)])
def test_exact_sums_of_squares(m, variant, ksplit, n):
    """Statistics kept as exact sums: equal integers from every launch, the float64 sum of the stored values but for
    the tiles' fp32 rounding (16 values each: under 2^-20), and, read back, the bits of the same value as a float."""
    torch.manual_seed(m)
    k = 4096
    w, up = (D.PackedWeight(torch.randn(*s, device=DEV).bfloat16()) for s in ((n, k), (512, n)))
    x = torch.randn(m, k, device=DEV).bfloat16()
    y = torch.randn(m, n, device=DEV).bfloat16()
    x[:5] = 0  # these rows' residual stays what it is
    y[0], y[1], y[2, ::3], y[3, 7], y[4, 9] = 0, 1e-20, 1e15, 1e20, float("nan")
    got = []
    for _ in range(4):
        sums, old, out = *torch.zeros(2, D.SUM_WORDS, m, dtype=torch.int64, device=DEV), y.clone()
        old.fill_(7)
        D.skinny_gemm(x, w, out=out, resid_ss=sums, zero=old, variant=variant, ksplit=ksplit)
        assert not old.any()
        got.append(sums)
    assert all(torch.equal(got[0], g) for g in got)
    value = [_exact(r) for r in got[0].T.tolist()]
    want = out.double().pow(2).sum(-1).tolist()
    assert value[0] == 0 and value[3] == float("inf") and value[4] != value[4]
    for i in (1, 2, *range(5, m)):
        assert abs(value[i] - want[i]) <= 2.0 ** -20 * want[i], i
    a, b = (D.skinny_gemm(out, up, rms=r) for r in (got[0], torch.tensor(value, dtype=torch.float32, device=DEV)))
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    with pytest.raises(ValueError):
        D.skinny_gemm(x, w, out=out, resid_ss=got[0], zero=torch.zeros(m, device=DEV))
    with pytest.raises(ValueError):
        D.skinny_gemm(out, up, rms=got[0][:, :m - 1].contiguous())


@pytest.mark.gpu
@pytest.mark.parametrize("m", [129, 160, 241, 256])
@pytest.mark.parametrize("ks", [1, 2, 7])
def test_plain_products_above_128_rows_store_what_the_epilogues_do(m, ks):
    """They have a way out of their own; the general one with a row scale of one gives the same bits, and rows and
    columns outside the output stay as they were."""
    n, k = 256, 512 * ks
    x, w = (torch.rand(r, k, device=DEV) * 2 - 1 for r in (m, n))
    pw, x, ss = D.PackedWeight(w.bfloat16()), x.bfloat16(), torch.full((m,), float(k), device=DEV)
    for v in D.skinny_variants(m):
        buf = torch.full((m + 1, n + 8), 7.0, device=DEV, dtype=torch.bfloat16)
        D.skinny_gemm(x, pw, out=buf[:m, :n], variant=v, ksplit=ks)
        want = x.double() @ w.bfloat16().double().T
        # rsqrt(k * (1 / k)) is exactly one for powers of two
        scaled = D.skinny_gemm(x, pw, rms=ss, eps=0.0, variant=v, ksplit=ks)
        if k & (k - 1) == 0:
            assert torch.equal(buf[:m, :n], scaled)
        assert float((buf[:m, :n].double() - want).norm() / want.norm()) < 2.0 ** -8
        assert bool((buf[m] == 7).all()) and bool((buf[:, n:] == 7).all())
