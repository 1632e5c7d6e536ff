"""Decode-path ops on ``native/kernels/decode.hip`` -- the one-token-per-sequence
half of LLM serving, which is HBM-bound on the weights and the KV cache.

* :func:`pack_weight` / :class:`PackedWeight` -- a ``[N, K]`` bf16 weight
  rearranged ONCE into MFMA A-fragment order (``[N/16][K/32][64][8]``), so the
  skinny GEMM streams it as contiguous 1 KB wave loads straight into registers.
* :func:`skinny_gemm` -- ``x[M, K] @ W^T`` for a decode batch ``M <= 256``
  (split-K with an in-kernel last-arriver reduction when ``N`` is small).
* :class:`PagedKVCache` -- ``[layers, pages, kv_heads, K|V, 32 x 128]`` bf16
  pages whose element order IS the MFMA operand order of the decode attention
  (:func:`kv_index_tables`); a 32-token page of one KV head is 16 KB.
* :func:`rope_cache_` -- RoPE on the q/k heads of fused QKV rows + scatter of k/v
  into their cache slots, one launch.
* :func:`paged_decode_attention` -- GQA decode attention over the paged cache
  (context split across waves, log-sum-exp merge by the last split, one launch).

Every op raises :class:`kgs.ops.NativeUnavailable` when the native library is
missing; the ``ref_*`` functions are the plain-PyTorch fp32 references (they run
on CPU too and define the cache layout for tests).
"""
from __future__ import annotations

import math
from functools import lru_cache
import os

import torch

from . import _lib
from .activation import Gate

PAGE = 32
HEAD_DIM = 128
CUS = 256  # MI355X compute units (grid sizing)


# ----------------------------------------------------------------------------
# weights

def pack_weight(w: torch.Tensor) -> torch.Tensor:
    """``[N, K]`` -> ``[N/16, K/32, 64, 8]``: lane ``g*16 + r`` of fragment
    ``(nt, kk)`` holds ``W[16 nt + r, 32 kk + 8 g : +8]`` (16x16x32 bf16 A map)."""
    n, k = w.shape
    if n % 16 or k % 32:
        raise ValueError(f"pack_weight needs N % 16 == 0 and K % 32 == 0, got {tuple(w.shape)}")
    return w.reshape(n // 16, 16, k // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous()


def unpack_weight(p: torch.Tensor) -> torch.Tensor:
    nt, kk = p.shape[:2]
    return p.reshape(nt, kk, 4, 16, 8).permute(0, 3, 1, 2, 4).reshape(nt * 16, kk * 32)


def swiglu_rows(n2: int) -> torch.Tensor:
    """Row order of a fused gate|up weight ``[2I, K]`` (gate rows first) in which
    16-row tile ``t`` holds gate rows ``8t..8t+7`` then up rows ``8t..8t+7``: the
    skinny GEMM's SwiGLU epilogue pairs them lane-to-lane (``lane ^ 32``)."""
    if n2 % 32:
        raise ValueError("fused gate|up weight needs 2I % 32 == 0")
    inter = n2 // 2
    return torch.arange(n2).reshape(2, inter // 8, 8).permute(1, 0, 2).reshape(n2)


def rope_rows(n: int, heads: int, kv_heads: int) -> torch.Tensor:
    """Row order of a fused qkv weight ``[(H + 2 HKV) * 128, K]`` in which every
    q / k head's 16-row tile ``t`` holds dims ``8t..8t+7`` then ``64+8t..64+8t+7``
    (v heads unchanged): the skinny GEMM's RoPE epilogue pairs each rotate-half
    partner lane-to-lane (``lane ^ 32``)."""
    if n != (heads + 2 * kv_heads) * HEAD_DIM:
        raise ValueError(f"qkv weight of {n} rows does not match {heads} + 2 x {kv_heads} heads of {HEAD_DIM}")
    head = torch.arange(HEAD_DIM).reshape(2, 8, 8).permute(1, 0, 2).reshape(HEAD_DIM)
    rot = heads + kv_heads
    q_k = (torch.arange(rot)[:, None] * HEAD_DIM + head[None, :]).reshape(-1)
    return torch.cat([q_k, torch.arange(rot * HEAD_DIM, n)])


def pack_swiglu(w: torch.Tensor) -> torch.Tensor:
    return pack_weight(w[swiglu_rows(w.shape[0]).to(w.device)])


FP8 = torch.float8_e4m3fn
FP8_MAX = 448.0


class PackedWeight:
    """A projection weight in skinny-GEMM fragment order (plus its shape).

    * ``swiglu=True``: a fused gate|up weight whose GEMM emits ``act(g) * u``
      (``act``: ``"silu"``, ``"gelu_tanh"`` or a :class:`kgs.ops.activation.Gate`);
    * ``fold``: an RMSNorm weight ``[K]`` folded into the columns (``W * fold``),
      for GEMMs that apply the norm in their epilogue (``rms=``);
    * ``fp8=True``: weight-only fp8 (W8A16): OCP e4m3 with one scale per output
      row, dequantised to bf16 in registers (half the HBM bytes per step);
    * ``rope=(H, HKV)``: a fused qkv weight in :func:`rope_rows` order, for the
      GEMM whose epilogue applies RoPE and writes the KV cache (``rope=`` of
      :func:`skinny_gemm`); its output is in the original order."""

    __slots__ = ("data", "n", "k", "swiglu", "fp8", "wscale", "rope", "act")

    def __init__(self, w: torch.Tensor, swiglu: bool = False, fold: torch.Tensor | None = None, fp8: bool = False,
                 rope: tuple | None = None, act="silu"):
        self.n, self.k = w.shape
        self.act = Gate.of(act)
        self.swiglu, self.fp8, self.rope = swiglu, fp8, rope
        if swiglu and rope:
            raise ValueError("a weight is either SwiGLU- or RoPE-packed")
        rows = swiglu_rows(self.n).to(w.device) if swiglu else \
            rope_rows(self.n, *rope).to(w.device) if rope else None
        if fold is not None:
            w = w.float() * fold.float()[None, :]
        if fp8:
            wf = w.float()
            scale = wf.abs().amax(1).clamp(min=1e-12) / FP8_MAX
            q = (wf / scale[:, None]).clamp(-FP8_MAX, FP8_MAX).to(FP8).view(torch.uint8)
            if rows is not None:
                q, scale = q[rows], scale[rows]
            self.data = pack_weight(q)
            self.wscale = scale.float().contiguous()
        else:
            w = w.to(torch.bfloat16)
            self.data = pack_weight(w[rows] if rows is not None else w)
            self.wscale = None

    @property
    def n_out(self) -> int:
        return self.n // 2 if self.swiglu else self.n

    def unpacked(self) -> torch.Tensor:
        """The weight as the kernel sees it (dequantised for fp8), in original row order."""
        p = unpack_weight(self.data)
        if self.fp8:
            p = (p.view(FP8).float() * self.wscale[:, None]).to(torch.bfloat16)
        if self.swiglu or self.rope:
            rows = swiglu_rows(self.n) if self.swiglu else rope_rows(self.n, *self.rope)
            inv = torch.empty(self.n, dtype=torch.long, device=p.device)
            inv[rows.to(p.device)] = torch.arange(self.n, device=p.device)
            p = p[inv]
        return p


# tile variants of native/kernels/decode.hip (id -> (R W-row tiles per wave,
# MT 16-column x tiles, KC k-steps per x chunk)); 0 = default for the batch size
SKINNY_VARIANTS = {
    1: (1, 1, 16), 2: (1, 1, 8), 3: (2, 1, 16),
    4: (1, 2, 16), 5: (1, 2, 8), 6: (2, 2, 8), 7: (2, 2, 16),
    8: (1, 4, 16), 9: (1, 4, 4), 10: (1, 4, 8), 11: (2, 4, 4), 12: (2, 4, 8),
    13: (2, 8, 2), 14: (2, 8, 4), 15: (4, 8, 2), 16: (1, 8, 4),
    17: (2, 16, 2), 18: (1, 16, 4), 19: (1, 16, 2),
    20: (1, 1, 8), 21: (2, 1, 8), 22: (1, 2, 8), 23: (2, 2, 8), 24: (1, 4, 8), 25: (2, 4, 8),
}
# variants whose four waves split one strip's K range (decode.hip skinny KIN):
# strips of 16 R rows, chunks of 4 x KC k-steps, no cross-workgroup split-K
KIN_VARIANTS = frozenset({20, 21, 22, 23, 24, 25})
_DEFAULT_VARIANT = {1: 1, 2: 4, 4: 8, 8: 13, 16: 17}

# Measured routing per (MT, N, K) on MI355X with weights streamed from HBM
# (bench/decode_bench.py --tune, profiles/decode_tune.md): (variant, ksplit) of
# the skinny GEMM where it beat hipBLASLt, None where hipBLASLt won. Shapes:
# Llama-3-8B qkv 6144x4096, o 4096x4096, gate|up 28672x4096, down 4096x14336,
# lm_head 128256x4096.
_QKV, _O, _GU, _DOWN, _LM = (6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336), (128256, 4096)
TUNED: dict = {
    (1, *_QKV): (1, 2), (1, *_O): (20, 1), (1, *_GU): (3, 1), (1, *_DOWN): (1, 4), (1, *_LM): (1, 1),
    (2, *_QKV): (4, 2), (2, *_GU): (6, 1), (2, *_DOWN): (4, 4), (2, *_LM): (6, 1),
    (4, *_QKV): None, (4, *_O): (9, 4), (4, *_GU): (11, 1), (4, *_DOWN): (10, 4), (4, *_LM): (11, 1),
    (8, *_QKV): None, (8, *_O): None, (8, *_GU): None, (8, *_DOWN): (16, 4), (8, *_LM): None,
    (16, *_QKV): None, (16, *_O): None, (16, *_GU): None, (16, *_DOWN): None, (16, *_LM): None,
}
# few-row batches: (variant, ksplit, up to M) -- the in-workgroup K split
# (variant 20) wins while x is a few rows (each wave reads its B fragments
# straight from L2, so x traffic grows with M); profiles/r2/skinny_kin_tune.jsonl
TUNED_TINY: dict = {_QKV: (20, 1, 8), _GU: (20, 1, 4), _DOWN: (20, 1, 2)}
TUNED_TINY_FP8: dict = {_GU: (21, 1, 4), _DOWN: (21, 7, 4)}
# the same sweep for weight-only fp8 (--tune --fp8): (variant, ksplit) per (MT, N, K)
TUNED_FP8: dict = {
    (1, *_QKV): (20, 1), (2, *_QKV): (5, 4), (4, *_QKV): (9, 4),
    (1, *_O): (20, 1), (2, *_O): (5, 4), (4, *_O): (10, 4),
    (1, *_GU): (1, 1), (2, *_GU): (7, 1), (4, *_GU): (12, 2),
    (1, *_DOWN): (1, 7), (2, *_DOWN): (5, 8), (4, *_DOWN): (9, 8),
    (1, *_LM): (1, 1), (2, *_LM): (6, 1), (4, *_LM): (11, 1),
}
# Decode batches above the fused range: K slices of the split-K 256x256 GEMM
# (kgs.ops.gemm.gemm_nt_splitk) per (batch bucket, N, K) where it beat both
# hipBLASLt and the skinny GEMM (bench/decode_bench.py --wide,
# profiles/decode_wide_gemm.jsonl): down 1.89x / 1.14x / 1.48x at 128 / 256 /
# 512, qkv 1.22x at 256, o 1.07x at 128. gate|up (fp32 partials too large) and
# the rest stay on hipBLASLt.
SPLITK_TUNED: dict = {
    (128, *_DOWN): 16, (128, *_O): 8,
    (256, *_QKV): 8, (256, *_DOWN): 8,
    (512, *_DOWN): 8,
    # Llama-3-70B (decode without packed copies, `--model llama3-70b`; bench/decode_bench.py --wide
    # --model llama3-70b): down 1.55x / 1.83x / 2.3x at 64 / 128 / 256, qkv 1.40x and o 1.47x at 256;
    # 1 = the plain 256x256 GEMM (gate|up at 256: 1.22x)
    (64, 8192, 28672): 8,
    (128, 10240, 8192): 4, (128, 8192, 8192): 8, (128, 8192, 28672): 8,
    (256, 10240, 8192): 4, (256, 8192, 8192): 8, (256, 8192, 28672): 8, (256, 57344, 8192): 1,
}
SPLITK_WS_FLOATS = 8 * 256 * 8192  # the largest entry above (M x N x slices)

# Decode batches 49-512 on the four-wave kernel (kgs.ops.gemm.gemm_nt_w4x):
# (tile width, K slices, tile height) per (batch bucket, N, K) where it beat
# hipBLASLt and the 8-wave split-K, weights streamed from HBM
# (bench/decode_w4x_sweep.py, profiles/r2/decode_w4x_sweep.jsonl and
# decode_w4x_bm128.jsonl, decode_w4x_lm_head.jsonl; speed-up vs hipBLASLt in the comments). Batches up to
# 128 take 128-row tiles (no MFMAs on padding rows: qkv / o / down 3-20 %
# faster than 256-row tiles at 64-128 rows, and ahead of the fused skinny
# GEMMs from 49 rows up). Buckets not listed stay on the routes below.
_W4X_BUCKETS = (64, 96, 128, 192, 256, 384, 512)
W4X_MIN_BATCH = 49
W4X_TUNED: dict = {
    (64, *_QKV): (128, 4, 128), (96, *_QKV): (128, 8, 128), (128, *_QKV): (128, 4, 128),  # 1.99/4.39/3.31
    (64, *_O): (128, 8, 128), (96, *_O): (128, 8, 128), (128, *_O): (128, 8, 128),  # 4.95/2.27/2.22
    (64, *_GU): (128, 1, 128), (96, *_GU): (128, 1, 128), (128, *_GU): (128, 1, 128),  # 1.16/1.15/1.14
    (64, *_DOWN): (128, 8, 128), (96, *_DOWN): (128, 8, 128), (128, *_DOWN): (128, 8, 128),  # 1.75/2.07/2.29
    (64, *_LM): (256, 1, 128), (96, *_LM): (256, 1, 128), (128, *_LM): (256, 1, 128),  # 1.18/1.22/1.24
    (192, *_QKV): (128, 4, 256), (256, *_QKV): (128, 4, 256), (384, *_QKV): (128, 2, 256),  # 1.39/1.49/1.06
    # o at 192-256 rows: 128-row tiles, 4 slices (half the fp32 partials of 256-row tiles x 8 slices;
    # probe 29.6 / 30.6 vs 32.9 / 33.7 us, serving b256 +0.8 % A/B/A, profiles/r3/decode/route_ab)
    (192, *_O): (128, 4, 128), (256, *_O): (128, 4, 128), (384, *_O): (128, 4, 256),  # -/-/1.02
    (512, *_O): (128, 4, 256),  # 1.10
    (192, *_GU): (128, 1, 256), (256, *_GU): (128, 1, 256), (512, *_GU): (256, 1, 256),  # 1.07/1.06/1.06
    (192, *_DOWN): (128, 8, 256), (256, *_DOWN): (128, 8, 256), (384, *_DOWN): (128, 4, 256),  # 2.7/1.5/1.4
    (512, *_DOWN): (128, 4, 256),  # 1.45
}


def _apply_w4x_override(spec: str) -> None:
    """``KGS_W4X_ROUTES="256,4096,4096=128,4,128,4;..."``: (bucket, N, K) =
    (bn, slices, bm[, stages]) entries replacing W4X_TUNED's, for same-box
    routing A/B runs (scripts/gpu.sh route_ab); ``=none`` removes an entry."""
    for item in filter(None, (s.strip() for s in spec.split(";"))):
        key, _, val = item.partition("=")
        k = tuple(int(t) for t in key.split(","))
        if len(k) != 3 or k[0] not in _W4X_BUCKETS:
            raise ValueError(f"KGS_W4X_ROUTES: bad key {key!r}")
        if val.strip() == "none":
            W4X_TUNED.pop(k, None)
            continue
        v = tuple(int(t) for t in val.split(","))
        if len(v) not in (3, 4):
            raise ValueError(f"KGS_W4X_ROUTES: bad route {val!r}")
        W4X_TUNED[k] = v


if os.environ.get("KGS_W4X_ROUTES"):
    _apply_w4x_override(os.environ["KGS_W4X_ROUTES"])


def w4x_route(m: int, n: int, k: int):
    """(tile width, K slices, tile height[, LDS stages]) of the four-wave
    decode GEMM for batch m, or None. The tuple's order is
    ``gemm_nt_w4x_partials``'s (bn, nslice, bm, stages) positional order."""
    if m < W4X_MIN_BATCH or m > 512:
        return None
    b = next(x for x in _W4X_BUCKETS if m <= x)
    return W4X_TUNED.get((b, n, k))


W4X_RULE_MIN = 33   # rows: skinny GEMM below
W4X_RULE_MAX = 256


def w4x_rule(m: int, n: int, k: int, most: int = 16, cus: int = CUS):
    """The route (as :func:`w4x_route`) for 33 to 256 rows of a size without measured entries, or None.
    ``most``: slices that the caller can take.

    128x128 tiles in as many K slices (of at least 256) as fit one workgroup on every CU: a
    second round of workgroups costs more than finer slices give, wider tiles leave
    CUs idle. Tiles of 256 rows only where 128-row ones alone are more than the CUs. us at 100
    rows, weights from HBM, next to the library's product: 3072x2048 8.5 / 12.4 (with 4 slices
    9.5, with 16 12.8), 2048x2048 7.4 / 11.2, 16384x2048 17.7 / 21.0 (unsplit 24.4), 2048x8192 12.6 /
    21.2 (8 slices 15.2), 32000x2048 30.5 / 33.1; at 256 rows 2048x8192 18.0 / 27.2, 16384x2048 25.6 /
    30.1. The slices' sum is left to the norm, rotation or gate that follows; a launch of its own for
    it costs 3 to 6 us more, and 16 slices there more than they give (``most`` = 8). None where the tiles are more
    than the CUs, or a K like 11008 that slices badly leaves half of the CUs idle."""
    if not W4X_RULE_MIN <= m <= W4X_RULE_MAX or n % 128 or k % 128 or (n, k) in _MEASURED:
        return None
    bm = 128 if -(-m // 128) * (n // 128) <= cus else 256
    tiles = -(-m // bm) * (n // 128)
    ns = 1
    while 2 * ns <= most and 2 * ns * tiles <= cus and k % (256 * ns) == 0 and k >= 512 * ns:
        ns *= 2
    if tiles > cus or (2 * ns * tiles < cus and k >= 512 * ns and 2 * ns <= most):
        return None
    return 128, ns, bm


def gate_rule(m: int, n: int, k: int, sliced: bool) -> int | None:
    """Rows (64 or 128) of the gate kernel's tiles (:func:`kgs.ops.gemm.gemm_gate`) for a fused gate|up of ``n`` rows at up to 128
    rows, None where 128-wide tiles are faster, or (``sliced``: the caller has a route of K slices) those in slices.

    Its tiles of 32 outputs are a workgroup for every CU at n = 16384 and half of them or fewer rows below; up to 64 rows
    two share a CU. us in a chain of launches, weights from HBM, 128-wide tiles in slices with their sum / without / so: 16384x2048
    at 36 rows 20.0 / 24.1 / 17.5, 100 23.6 / 25.6 / 19.9, 8192x2048 at 100 18.2 / 23.4 / 13.7, 16384x4096 42.8 / 44.7 / 33.9, 11008x2048
    at 64 19.3 / 23.2 / 15.3; without slices 28672x4096 at 64 58.6 / 51.3, 24576x2048 28.2 / 27.9, but 32768x2048 37.6 / 39.6 and at
    100 rows 22016x4096 52.5 / 61. A long sum on less than half of the CUs, or from 65 rows on on less than seven eighths, is
    better in slices: 8192x4096 at 64 21.5 / 24.8, 6144x6144 27.0 / 37.6, 10240x5120 at 96 43.0 / 45.9."""
    wgs = -(-(n // 2) // 32)
    if not 0 < m <= 128 or n % 16 or k % 8 or wgs > (448 if m <= 64 else CUS):
        return None
    if sliced and ((2 * wgs <= CUS and k > 2048) or (m > 64 and 8 * wgs < 7 * CUS and k > 4096)):
        return None
    return 64 if m <= 64 or 2 * wgs <= CUS else 128


_MEASURED = {key[1:] for key in (*W4X_TUNED, *SPLITK_TUNED)}


def w4x_stages(route) -> int:
    """LDS stages that a W4X_TUNED route asks for (2 unless the entry names 3 or 4; tiles smaller than 256x256 run on three or four in any case)."""
    return route[3] if len(route) > 3 else 2


# Decode weights are read once per step by one CU each: their loads go
# non-temporal (gemm_w4.h AUX 52, B's loads only; the activations, re-read by
# every workgroup from L2, keep the default policy). gate|up at batch 256:
# 69.1 -> 68.0 us row-major, 67.5 -> 64.9 us tile-panel packed
# (profiles/r4/decode/README.md); batch-256 serving, two A/B/A passes on one
# box: 18 247 -> 18 302 output tok/s (profiles/r5/decode/README.md). On by
# default since round 5: the fault that kept it opt-in in round 4 was the
# graph memset node of the persistent GEMM's ticket slot, not these loads
# (profiles/r5/fault/README.md; the nt kernels differ from the default ones
# only in the nt bit of B's buffer loads). KGS_NT_WEIGHTS=0 turns it off.
NT_WEIGHTS = os.environ.get("KGS_NT_WEIGHTS", "1") == "1"


def w4x_nt(route) -> bool:
    """Stream this route's weights non-temporally (two-stage routes only)."""
    return NT_WEIGHTS and w4x_stages(route) == 2


def w4x_split_bns(n: int, k: int) -> set:
    """Tile widths the split-K four-wave routes use for an ``[n, k]`` weight
    (the bn a tile-panel copy must be packed with)."""
    return {r[0] for (_, rn, rk), r in W4X_TUNED.items() if (rn, rk) == (n, k) and r[1] > 1}


def splitk_slices(m: int, n: int, k: int) -> int | None:
    """K slices for a decode GEMM of batch m (bucketed to a power of two), or
    None when the split-K kernel is not the measured winner."""
    mb = 1 << max(0, (m - 1).bit_length())
    return SPLITK_TUNED.get((mb, n, k))


SKINNY_DEFAULT_MAX_M = 32  # untuned shapes: skinny GEMM up to this batch, hipBLASLt above


def _mt(m: int) -> int:
    if not 0 < m <= 256:
        raise ValueError(f"skinny GEMM batch must be 1..256, got {m}")
    return 1 if m <= 16 else 2 if m <= 32 else 4 if m <= 64 else 8 if m <= 128 else 16


def skinny_variants(m: int) -> list[int]:
    mt = _mt(m)
    return [v for v, (_, vmt, _) in SKINNY_VARIANTS.items() if vmt == mt]


def skinny_geometry(m: int, variant: int = 0) -> tuple[int, int, int]:
    """(rows of W per workgroup strip, k per x chunk, padded batch) -- mirrors
    ``kgs_skinny_variant_geometry`` in decode.hip."""
    mt = _mt(m)
    v = variant or _DEFAULT_VARIANT[mt]
    r, vmt, kc = SKINNY_VARIANTS[v]
    if vmt != mt:
        raise ValueError(f"variant {variant} is for {16 * vmt}-column batches, not M={m}")
    if v in KIN_VARIANTS:
        return 16 * r, 128 * kc, 16 * mt
    return 64 * r, 32 * kc, 16 * mt


def choose_ksplit(m: int, n: int, k: int, cus: int = CUS, variant: int = 0) -> int:
    """Largest divisor of the k-chunk count that keeps the grid within one
    workgroup per CU (measured best: long-running streaming workgroups,
    profiles/decode_kernels.md) and the fp32 slabs within 64 MB (1 = no split)."""
    rps, kpc, mpad = skinny_geometry(m, variant)
    nstrip, nchunks = n // rps, k // kpc
    best = 1
    for d in range(2, nchunks + 1):
        if nchunks % d:
            continue
        if nstrip * d > max(cus, nstrip) or d * mpad * n * 4 > (64 << 20):
            break
        best = d
    return best


@lru_cache(maxsize=4096)
def skinny_rule(m: int, n: int, k: int, one: bool = False) -> tuple[int, int]:
    """(variant, ksplit) of bf16 weights without a measured entry; ``one``: one W-row tile per wave.

    The K split inside the workgroup (16 rows of W each, no slabs in memory and no ticket, 2 to 3 us
    of a launch) where its strips are a workgroup per CU or so: up to 6144 rows, two tiles a wave
    above 4096 from 17 rows of x on; at 17 to 32 rows of x and K up to 2048 to 8192, one round of two-tile workgroups (us at 24 rows, slabs /
    so: 8192x2048 13.5 / 10.9, 6656x2048 13.2 / 11.1, 8192x1024 10.2 / 7.0; 10240x2048, where it is a second round, 13.5 / 14.3), in one tile a wave (``one``: weights packed with
    RoPE), which is a second round there, up to 48k values of x (17 rows of 8192x2048 13.8 / 11.1, 24 14.0 / 13.5, 32 14.0 / 14.7; 32 of x1024 10.7 / 8.7). Every workgroup reads all of x, which bounds K by the rows: up to 16 rows K of
    8192 (in two halves where that is no second round of workgroups; else, from 64k values of x on, only where slabs
    would not fill three quarters of the CUs), of 32k values where the strips are more than the CUs; up to 32 rows K of
    4096 (96k values on less than half of the CUs and in two tiles a wave); beyond them 160k values; from 17 rows on
    K of 2048 where two tiles a wave leave more than a quarter of the CUs idle. us at 24 rows, before /
    so: 3072x2048 10.3 / 6.9, 2048x2048 9.4 / 6.7, 6144x2048 12.4 / 9.9, 4096x4096 14.3 / 11.5; at 1 row 7.6 /
    5.0, 6.9 / 4.7, 9.7 / 6.9; at 64 rows 2048x2048 13.7 / 11.7, but 4096x4096 18.2 / 20.8; at 16 rows 5120x3072
    10.9 / 13.2 and 3072x8192 14.6 / 16.0 (18.3 in halves), at 32 5120x3072 13.2 / 14.5 and 1024x4096 11.6 / 12.5.
    Else x chunks of 8 k-steps instead of 16 from 17 rows on (16384x2048 at 40 rows 22.8 / 18.5,
    32000x2048 42 / 31), but not up to 32 rows where a grid short of the CUs has 2048 and more of K in a workgroup
    (5120x10240 at 24 rows 30.2 / 32.2, 9216x3072 17.8 / 18.6), and not in more slices than with 16 where those are
    shorter than 512 (1024x4096 at 48 rows 15.5 / 18.0 in 16 slices; 3584x3584 at 24 in one 18.9, in two 15.1)."""
    mt = _mt(m)
    strips = n // 16
    if mt <= 4 and k % 1024 == 0 and n % 32 == 0 and strips <= (512 if mt == 2 and k <= 2048 and (not one or m * k <= 48 << 10) else 384):
        over = strips > CUS
        wide = mt > 1 and over and not one
        v = {1: 20, 2: 23 if wide else 22, 4: 25 if wide else 24}[mt]
        if mt == 1 and k <= 8192 and (not over or m * k <= 32 << 10):
            halves = k > 4096 and 2 * strips <= CUS and k % 2048 == 0
            if halves or k <= 4096 or m * k <= 64 << 10 or 4 * (n // 64) * choose_ksplit(m, n, k) < 3 * CUS:
                return v, 2 if halves else 1
        if not over or k <= 2048 or (wide and 4 * (strips // 2) >= 3 * CUS):
            if mt == 2 and k <= 4096 and (m * k <= 96 << 10 or (2 * strips >= CUS and not wide)):
                return v, 1
            if mt == 4 and m * k <= 160 << 10:
                return v, 1
    v = {2: 5, 4: 10}.get(mt, _DEFAULT_VARIANT[mt])
    ks = choose_ksplit(m, n, k, variant=v)
    if mt in (2, 4) and k % 512 == 0:
        coarse = choose_ksplit(m, n, k)
        if mt == 2 and ks == coarse and k // ks >= 2048 and n // 64 * ks < CUS:
            v = _DEFAULT_VARIANT[mt]
        elif ks > coarse and k // ks < 512:
            ks = coarse
    return v, ks


def skinny_config(m: int, n: int, k: int, fp8: bool = False) -> tuple[int, int]:
    """(variant, ksplit) for a skinny-GEMM call: the tuned entry, else by rule."""
    tiny = (TUNED_TINY_FP8 if fp8 else TUNED_TINY).get((n, k))
    if tiny is not None and m <= tiny[2]:
        return tiny[:2]
    hit = (TUNED_FP8 if fp8 else TUNED).get((_mt(m), n, k))
    if hit is not None:
        return hit
    if not fp8:
        return skinny_rule(m, n, k)
    v = _DEFAULT_VARIANT[_mt(m)]
    return v, choose_ksplit(m, n, k, variant=v)


def _skinny_plan(m: int, n: int, k: int, fp8: bool, rope: bool) -> tuple[int, int]:
    variant, ks = skinny_config(m, n, k, fp8=fp8)
    if rope and SKINNY_VARIANTS[variant][0] != 1:
        # the RoPE epilogue is built for one-tile waves (R 1)
        variant, ks = skinny_rule(m, n, k, one=True)
    return variant, ks


@lru_cache(maxsize=4096)
def skinny_takes(m: int, n: int, k: int, fp8: bool = False, rope: bool = False) -> bool:
    """Whether :func:`skinny_gemm` runs ``m`` rows of an ``[n, k]`` weight: up to 256 (64 of an e4m3 weight, and of a
    RoPE-packed one, whose epilogue is built for these), on the strips and chunks of its choice."""
    if not 0 < m <= (64 if fp8 or rope else 256):
        return False
    strip, chunk, _ = skinny_geometry(m, _skinny_plan(m, n, k, fp8, rope)[0])
    return n % strip == 0 and k % chunk == 0


def use_skinny(m: int, n: int, k: int) -> bool:
    """Decode routing: True = skinny GEMM, False = the library GEMM (hipBLASLt)."""
    if not 0 < m <= 256:
        return False
    key = (_mt(m), n, k)
    if key in TUNED:
        return TUNED[key] is not None
    return m <= SKINNY_DEFAULT_MAX_M


_WS: dict = {}
# Workspaces replaced by larger ones. hipGraphs captured before the growth still
# hold the old device pointers, so the old buffers must outlive them: they are
# kept here for the life of the process instead of going back to the caching
# allocator (where they could be reused, or released to the driver and fault).
_RETIRED: list = []


def device_key(device: torch.device) -> int:
    """Normalised per-GPU cache key: torch.device("cuda") and "cuda:0" differ as
    dict keys but name the same workspace."""
    return device.index if device.index is not None else torch.cuda.current_device()


def retire(*bufs) -> None:
    _RETIRED.extend(b for b in bufs if b is not None)


def _workspace(device: torch.device, floats: int, ints: int):
    """Per-device split-K slab buffer and zeroed ticket counters (the kernel
    re-arms the counters it uses). GEMMs of one device are stream-ordered."""
    key = device_key(device)
    ws, cnt = _WS.get(key, (None, None))
    if ws is None or ws.numel() < floats:
        retire(ws)
        ws = torch.empty(max(floats, 1 << 20), dtype=torch.float32, device=device)
    if cnt is None or cnt.numel() < ints:
        retire(cnt)
        cnt = torch.zeros(max(ints, 4096), dtype=torch.int32, device=device)
    _WS[key] = (ws, cnt)
    return ws, cnt


EPI_SWIGLU, EPI_RMS, EPI_RESID, EPI_ROPE, EPI_GELU, EPI_CLAMPED, EPI_SUMS_IN, EPI_SUMS_OUT, EPI_OWN = 1, 2, 4, 8, 16, 32, 64, 128, 256
SUM_WORDS, SUM_MAX_N = 8, 8192  # integers of a row's exact sum of squares (decode.hip add_exact), longest row
GATE_EPI = {"silu": 0, "gelu_tanh": EPI_GELU, "clamped": EPI_CLAMPED}


@lru_cache(maxsize=4096)
def few_takes(m: int, n: int, k: int, fp8: bool = False, plain: bool = False) -> bool:
    """Whether the kernel of few rows (native/kernels/decode_few.hip) runs ``m`` rows of an ``[n, k]`` weight: up to 16 of bf16 weights (:func:`few_wide` has
    more), 32 of a product without a norm or a rotation (``plain``), which also takes any K of 64."""
    return not fp8 and 0 < m <= 32 and bool(_lib.lib().kgs_skinny_few_ok(m, n, k, plain))


@lru_cache(maxsize=4096)
def few_wide(m: int, n: int, k: int) -> bool:
    """Whether it takes 17 to 32 rows with a norm or a rotation too, and is the better one there: K of 1024 up to 8192, up to 16384 rows of W (us at 24 rows,
    others / so: 6144x4096 20.0 / 12.7, 2048x2048 7.6 / 5.8, 16384x2048 16.3 / 14.9; at 32 4096x14336 27.8 / 31.9, 28672x4096 42.6 / 46.6)."""
    return 16 < m <= 32 and n <= 16384 and k <= 8192 and bool(_lib.lib().kgs_skinny_few_wide_ok(m, n, k))


@lru_cache(maxsize=4096)
def few_route(m: int, n: int, k: int, plain: bool = False) -> bool:
    """Whether the kernel of few rows is the better one, of those that take these rows; us of plain products, weights from HBM, few / others.

    Beside :func:`skinny_gemm`: up to 8 rows where W is not much wider than the CUs are many (64000x1024 at 1 row 29 / 24.8, 64000x2048
    48.5 / 46.2, 32000x2048 23.8 / 23.0), beyond that from K = 3584 on up to 4 rows and where K is a multiple of 4096, whose strips lie at
    multiples of 128 KB, which skinny's four waves read at once (28672x4096 at 8 rows 36.2 / 41.6, 32000x4096 40.0 / 45.2). Not where W has as many strips
    at multiples of 256 KB as CUs (4096x8192 at 1 row 16.0 / 14.3, in two tiles a workgroup 8192x8192 at 8 31.8 / 28.3), nor short
    strips of long K, which skinny reads in slices (1024x14336 at 8 rows 16.9 / 13.4), nor a few more strips than CUs (5120x13824 at
    4 rows 30.3 / 28.0). Up to 16 rows while x is short, which every workgroup
    reads whole (6144x4096 at 16 11.0 / 13.6, but 2048x8192 12.7 / 11.6, 8192x7168 at 12 27 / 32), and of wide W where K is neither short nor long
    (28672x4096 at 12 37.8 / 42.1, 16384x2048 at 16 12.4 / 14.5, 32000x4096 42.0 / 46.2, but 32000x2048 26.7 / 23.5); up to 32
    for short K that does not divide by 1024 (24 rows: 2048x768 3.8 / 7.6, 4096x1536 6.7 / 9.6, but 2048x1024 5.5 / 4.6) and, with x by LDS,
    for K of 2048 to 8192 up to 8192 rows of W (24 rows: 2048x2048 5.5 / 6.9, 6656x2048 7.7 / 9.9).

    Beside the library, for sizes that skinny does not take: as long as neither x nor the grid is long (832x2048 at 1 row 3.6 / 7.9; 896x4864
    at 24 25.5 / 16.6, 13824x768 at 16 1.31 times its time, 6144x11008 1.15 times)."""
    if not few_takes(m, n, k, False, plain):
        return False
    if not (skinny_takes(m, n, k) if plain else _own_by_skinny(m, n, k, False, False)):
        if not plain:
            return True
        return n <= 32768 if m <= 8 else n <= 8192 and (n <= 4096 or k <= 8192) if m <= 16 else n <= 4096 and k <= 2048
    if m > 16:
        return (k <= 1536 and n <= 4096 and k % 1024 != 0) or (k >= 2048 and n <= 8192 and few_wide(m, n, k))
    if k % 8192 == 0 and ((n == 4096 and m <= 8) or (n == 8192 and m > 4)):
        return False
    if n <= 2048:
        return k <= (8192 if m <= 8 else 5120) or (k < 8192 and k % 1024 != 0)
    if m > 8:
        return m * k < 96 << 10 if n <= 8192 else k >= 2048 and (n <= 16384 or k >= 4096) and n <= 32768 and k <= 4096
    if 4096 < n <= 5120 and k > 8192 and k % 1024:
        return False
    if n <= 24576:
        return n <= 10240 or (k > 1024 and (m <= 4 or not 12288 < n < 16384))
    return (m <= 4 and k >= 3584) or k % 4096 == 0


@lru_cache(maxsize=4096)
def _own_by_skinny(m: int, n: int, k: int, fp8: bool, rope: bool) -> bool:
    v, ks = _skinny_plan(m, n, k, fp8, rope)
    return skinny_takes(m, n, k, fp8, rope) and not (ks > 1 and v in KIN_VARIANTS)


@lru_cache(maxsize=4096)
def own_takes(m: int, n: int, k: int, fp8: bool = False, rope: bool = False) -> bool:
    """Whether :func:`own_gemm` takes a norm in front of an ``[n, k]`` weight of ``m`` rows: up to 64 of bf16 weights that tile."""
    return not fp8 and 0 < m <= 64 and (few_takes(m, n, k) or _own_by_skinny(m, n, k, False, rope))


def own_gemm(x: torch.Tensor, w: PackedWeight, out: torch.Tensor | None = None, norm: bool = False, resid: bool = False,
             eps: float = 1e-5, rope: dict | None = None, counters: torch.Tensor | None = None) -> torch.Tensor:
    """:func:`skinny_gemm` with ``norm`` or ``resid``, by :func:`skinny_few` where that is the better one (:func:`few_route`)."""
    m, k = x.shape
    plain = not norm and rope is None
    # what skinny_gemm takes and skinny_few does not stays there: rows further apart than 32-bit offsets reach, an out of another shape; and what it refuses
    if not w.fp8 and few_wide(m, w.n, k) and x.stride(0) <= 1 << 25 and (out is None or out.shape == (m, w.n_out)) and not (norm and resid):
        return skinny_few(x, w, out, norm, resid, eps, rope)
    if m <= 16 and not w.fp8 and (few_route(m, w.n, k, plain) or (few_takes(m, w.n, k, False, plain) and not (
            skinny_takes(m, w.n, k) if plain else _own_by_skinny(m, w.n, k, False, bool(w.rope))))):
        return skinny_few(x, w, out, norm, resid, eps, rope)
    return skinny_gemm(x, w, out, norm=norm, resid=resid, eps=eps, rope=rope, counters=counters)


SLAB_ROWS = 96
WIDE_ROWS = 128


@lru_cache(maxsize=4096)
def slab_split(m: int, n: int, k: int, cus: int = CUS) -> tuple[int, int] | None:
    """(W tiles a wave, K slices) of :func:`skinny_slabs`, or None: up to 96 rows of W of 64 rows a workgroup (128 from N = 4096 on),
    in as many slices, 16 at most and of 128 at least, as leave one workgroup a CU, or half as many where :func:`_split` says so; the kernel then cuts W finer where that leaves CUs idle.
    us at 32 rows in 4 / 8 / 16 slices: 2048x8192 11.6 / 8.1 / 8.2, 4096x14336 27.0 / 19.6 / 21.6, 6144x4096 10.8 / 12.8 / -."""
    return _split(m, n, k, cus) if 0 < m <= SLAB_ROWS else None


@lru_cache(maxsize=4096)
def wide_split(m: int, n: int, k: int, cus: int = CUS) -> tuple[int, int] | None:
    """:func:`slab_split` of :func:`wide_slabs`, 97 to 128 rows. As many workgroups are the best there: us of the product alone at 128 rows in 2 / 4 / 8 / 16 slices 2048x2048 9.0 /
    6.7 / 6.5 / 8.4, 2048x8192 27.9 / 16.6 / 11.9 / 14.4, 6144x4096 by two tiles 23.6 / 17.1 / 20.3 (by one 18.6 in 2), 4096x14336 69 / 39.5 / 26.8 / 32.1."""
    return _split(m, n, k, cus) if SLAB_ROWS < m <= WIDE_ROWS else None


def _split(m: int, n: int, k: int, cus: int) -> tuple[int, int] | None:
    """(tiles of 64 rows to a strip, K slices). A slice more shortens the product and costs the launch that sums its parts, so the line lies where the two together are least.
    us of the product with the residual add and norm behind it, at 24 / 64 / 96 / 128 rows:

    * strips of 128 rows in 8 slices against strips of 64 in 4, as many workgroups: 4096x4096 13.2, 15.5, 17.7, 18.8 / 12.8, 13.9, 15.1, 16.8; 4096x2048 10.0, 13.0, 15.6, 18.0 /
      8.9, 10.7, 12.4, 14.0; 4096x8192 17.7, 20.7, 22.8, 23.4 / 16.9, 19.0, 21.6, 23.3; but 4096x14336 24.6, 27.6, 29.2, 31.6 / 25.1, 27.8, 30.8, 33.9, so up to K = 8192; and
      8192x8192 in 4 against 2 slices 30.1, 32.1, 33.9, 35.3 / 29.6, 30.7, 35.2, 39.5, so from 8 slices on;
    * strips of 64 rows in 8 slices against 4: 2048x2048 7.2, 9.1, 10.7, 12.2 / 7.3, 8.3, 9.5, 10.7; 2048x1024 6.3, 8.1, 9.5, 11.0 / 6.1, 7.1, 8.3, 9.5 (at 33 rows 7.9 / 7.7 and
      6.9 / 6.4, so above 32); but 2048x4096 8.9, 10.6, 12.1, 13.8 / 9.7, 10.9, 12.4, 14.1, so up to K = 2048; of 16 slices half as well (1024x2048 with a hyper-connection
      step behind it at 33 / 64 / 96 rows in 16, 8, 4: 7.9, 7.3, 7.9 / 9.3, 8.1, 8.3 / 10.9, 9.4, 9.5).

    The kernel sums the halves of such a slice apart, so that no chain is longer than those of the most slices."""
    r = 2 if n >= 4096 and n % 128 == 0 else 1
    if n <= 0 or k <= 0 or n % (64 * r) or k % 128:
        return None
    tiles, ns = n // (64 * r), 1
    while ns < 16 and 2 * ns * tiles <= cus and k % (256 * ns) == 0:
        ns *= 2
    if r == 2 and ns >= 8 and k <= 8192:
        return 1, ns // 2
    return r, ns // 2 if ns >= 8 and m > 32 and k <= 2048 else ns


@lru_cache(maxsize=4096)
def slab_rows_tiles(m: int, n: int, k: int, cus: int = CUS) -> int | None:
    """W tiles a wave of :func:`skinny_rows`, or None: two where 128 rows a workgroup are three quarters of the CUs or more (us at 48 rows with one /
    two: 28672x4096 48.0 / 39.8, 16384x2048 14.5 / 19.1; at 32 and fewer 32000x2048 23.4 / 28.3). The kernel takes strips between them where they fill the CUs better."""
    return _rows_tiles(m, n, k, cus) if 0 < m <= SLAB_ROWS else None


def _rows_tiles(m: int, n: int, k: int, cus: int) -> int | None:
    if n % 64 or k % 128:
        return None
    return 2 if m > 32 and n % 128 == 0 and 4 * (n // 128) >= 3 * cus else 1


@lru_cache(maxsize=4096)
def head_pays(m: int, n: int, k: int, cus: int = CUS) -> bool:
    """Whether 49 to 128 rows of an LM head on residual rows are better off on :func:`skinny_rows` (:func:`wide_rows`) than their norm's product
    with the rows of the weight: most of a round of workgroups or whole rounds, of K from 2048 on, where no four-wave tiles were measured to be better.
    us at 64 / 96 / 128 rows, four-wave tiles or the library / so: 32000x2048 32.2, 33.2, 34.5 / 29.3, 30.3, 30.9; 32000x4096 58.3, 58.6, 61.7 / 44.5, 46.7, 49.3;
    16384x2048 18.0, 19.0, 20.6 / 14.5, 16.0, 17.7; 64000x4096 119, 120, 121 / 86, 93, 100; not 32000x1024 15.7, 16.7, 17.5 / 15.7, 16.7, 17.6, nor 128256x4096,
    which has entries of its own, 181, 187, 190 / 187, 202, 214."""
    r = _rows_tiles(m, n, k, cus)
    if not 48 < m <= WIDE_ROWS or r is None or k < 2048 or w4x_route(m, n, k) is not None:
        return False
    wgs = n // (64 * r)
    rounds = -(-wgs // cus)
    return 20 * wgs >= 19 * rounds * cus if rounds > 1 else 4 * wgs >= 3 * cus


def rows_pay(m: int, n: int, k: int, gated: bool) -> bool:
    """Whether :func:`skinny_rows` beats what reads the weight's rows, by the time of the one over the other: of a gate and up at 17 to 32 rows one round
    of 64-row strips, or most of one of short K (16384x2048 0.93, 10240x2048 0.95, 10240x8192 1.04, 4096x4096 1.66); from 33 rows on its wide tiles in
    most of one round or in whole ones, of K that is worth a workgroup's start -- at 64 / 96 rows 28672x1024 1.18 / 1.19, x2048 1.04 / 1.07, 32000x2048 1.07 /
    1.11, x4096 0.92 / 0.97, 40960x4096 1.15 / 1.16, 64000x4096 0.91 / 0.96, 128256x4096, which has a measured entry, 1.03 / 1.13, 28672x6144 0.79 / 0.82; gated 28672x1536 0.97 / 1.07, x2048 1.01 / 1.04, x5120 0.84 / 0.92."""
    if m <= 32:
        return m > 16 and gated and k % 512 == 0 and slab_rows_tiles(m, n, k) is not None and \
            (56 * CUS < n <= 64 * CUS or (10240 <= n <= 56 * CUS and k <= 4096))
    if slab_rows_tiles(m, n, k) != 2:
        return False
    if gated:
        return k > 2048 if m <= 64 else k >= 5120
    wgs, rounds = n // 128, -(-n // (128 * CUS))
    if rounds > 1 and (20 * wgs < 19 * rounds * CUS or w4x_route(m, n, k) is not None):
        return False
    return k >= (3072 if m <= 64 or rounds == 1 else 5120)


@lru_cache(maxsize=4096)
def slabs_fill(m: int, n: int, k: int) -> bool:
    """Whether the slices of :func:`slab_split` are short or fill the CUs. A K like 11008 gives two slices of 43 ring rounds in a quarter of the workgroups
    that the CUs hold: the product and a hyper-connection step at 64 / 96 rows, over the general kernel's with the step, 4096x11008 1.65 / 1.82, 3072x14336 (slices of 3584,
    three quarters) 1.02 / 1.09, 5120x14336 (the same in wide tiles) 0.95 / 0.97, 2048x5632 (of 2816) 0.90 / 0.99."""
    split = slab_split(m, n, k)
    if split is None:
        return False
    r, ns = split
    wgs = n // (64 * r) * ns
    return wgs >= CUS or (wgs >= 48 and k // ns <= (4096 if r == 2 else 3072))


@lru_cache(maxsize=4096)
def slabs_pay(m: int, n: int, k: int) -> bool:
    """Whether a product left in slices to a hyper-connection step beats the whole product in front of it (times of both, in slices over whole): from 33 rows
    on where :func:`slabs_fill` says so. Up to 32 rows a product that one launch reads whole at full rate is better whole:
    of more than 2048 rows of W by the kernel of few rows (4096x4096 at 1 / 8 / 16 rows 1.23 / 1.24 / 1.15, 5120x2048 1.19 / 1.08 / 0.97, 2048x4096 0.94 / 0.89
    / 0.82), and of short K by skinny with K split in the workgroup (4096x1024 at 32 1.27, 4096x2048 1.09, 2048x1024 1.01); and so are two long
    slices in few workgroups (1024x13824 1.24 at 1 row, 4096x11008 1.23 at 32)."""
    split = slab_split(m, n, k)
    if split is None:
        return False
    if m > 32:
        return slabs_fill(m, n, k) and not (m > 64 and n >= 4096 and k <= 1024) and not (n > 4096 and k <= 512)
    r, ns = split
    if k // ns > 3072 and n // (64 * r) * ns < CUS // 2:
        return False
    if m <= 8:
        return not (k <= 1024 or (n > 2048 and k <= (8192 if m <= 4 else 7168)))
    if m <= 16:
        return not ((n >= 4096 and k <= 4096) or (n > 4096 and k <= 512))
    return not ((n >= 4096 and k in (1024, 2048)) or (n > 2048 and k <= 1024))


def _slab_operand(x: torch.Tensor, w: PackedWeight) -> tuple[int, int]:
    if x.dtype != torch.bfloat16 or not x.is_cuda or x.dim() != 2 or x.stride(1) != 1 or x.shape[1] != w.k:
        raise ValueError("x must be a row-major bf16 GPU matrix [M, K]")
    return x.shape


def skinny_slabs(x: torch.Tensor, w: PackedWeight) -> torch.Tensor:
    """``x @ W^T`` of up to 96 rows of a bf16 weight as fp32 parts ``[slices, M, N]`` of its sum, for a consumer that adds them
    (native/kernels/decode_slabs.hip; :func:`slab_split`). Columns in the order in which the weight is packed."""
    m, k = _slab_operand(x, w)
    return _slabs(x, w, m, k, slab_split, _lib.lib().kgs_skinny_slabs)


def wide_slabs(x: torch.Tensor, w: PackedWeight) -> torch.Tensor:
    """:func:`skinny_slabs` of 97 to 128 rows (:func:`wide_split`)."""
    m, k = _slab_operand(x, w)
    return _slabs(x, w, m, k, wide_split, _lib.lib().kgs_wide_slabs)


def _slabs(x, w, m, k, rule, kernel):
    split = None if w.fp8 or w.swiglu else rule(m, w.n, k)
    if split is None:
        raise ValueError(f"no slices for x {tuple(x.shape)}, W [{w.n}, {w.k}]")
    out = torch.empty((split[1], m, w.n), dtype=torch.float32, device=x.device)
    rc = kernel(w.data.data_ptr(), x.data_ptr(), out.data_ptr(), m, w.n, k, x.stride(0), *split, _lib.stream_handle(x.device))
    if rc:
        _lib.check(rc, f"slabs[{m}x{w.n}x{k}, {split}]")
    return out


def skinny_rows(x: torch.Tensor, w: PackedWeight, sq: torch.Tensor | None = None, eps: float = 1e-5) -> torch.Tensor:
    """``x @ W^T`` of up to 96 rows of a bf16 weight, or ``act(gate) * up`` of a gated one, by the kernel of :func:`skinny_slabs` in one slice;
    ``sq`` (fp32 ``[M]``): of x's RMSNorm (its weight folded into W) by these sums of squares of its rows."""
    m, k = _slab_operand(x, w)
    r = None if w.fp8 or w.rope else slab_rows_tiles(m, w.n, k)
    if r is None:
        raise ValueError(f"no tiles for x {tuple(x.shape)}, W [{w.n}, {w.k}]")
    if sq is not None and (sq.dtype != torch.float32 or sq.numel() != m or not sq.is_contiguous() or sq.device != x.device):
        raise ValueError("sq must be a contiguous fp32 vector, one a row of x")
    out = torch.empty((m, w.n_out), dtype=torch.bfloat16, device=x.device)
    rc = _lib.lib().kgs_skinny_rows(w.data.data_ptr(), x.data_ptr(), out.data_ptr(), m, w.n, k, x.stride(0), out.stride(0), r,
                                    EPI_SWIGLU | GATE_EPI[w.act.act] if w.swiglu else 0, None if sq is None else sq.data_ptr(),
                                    float(eps), w.act.limit, _lib.stream_handle(x.device))
    if rc:
        _lib.check(rc, f"skinny_rows[{m}x{w.n}x{k}]")
    return out


def wide_rows(x: torch.Tensor, w: PackedWeight, sq: torch.Tensor | None = None, eps: float = 1e-5) -> torch.Tensor:
    """:func:`skinny_rows` of 97 to 128 rows of a weight that is not gated."""
    m, k = _slab_operand(x, w)
    r = _rows_tiles(m, w.n, k, CUS) if SLAB_ROWS < m <= WIDE_ROWS and not (w.fp8 or w.rope or w.swiglu) else None
    if r is None:
        raise ValueError(f"no tiles for x {tuple(x.shape)}, W [{w.n}, {w.k}]")
    if sq is not None and (sq.dtype != torch.float32 or sq.numel() != m or not sq.is_contiguous() or sq.device != x.device):
        raise ValueError("sq must be a contiguous fp32 vector, one a row of x")
    out = torch.empty((m, w.n), dtype=torch.bfloat16, device=x.device)
    rc = _lib.lib().kgs_wide_rows(w.data.data_ptr(), x.data_ptr(), out.data_ptr(), m, w.n, k, x.stride(0), out.stride(0), r,
                                  None if sq is None else sq.data_ptr(), float(eps), _lib.stream_handle(x.device))
    if rc:
        _lib.check(rc, f"wide_rows[{m}x{w.n}x{k}]")
    return out


def rope_cache_packed(parts: torch.Tensor, sq: torch.Tensor, w: PackedWeight, eps: float, rope: dict) -> torch.Tensor:
    """The fused qkv rows ``[T, (H + 2 HKV) * 128]`` of a RoPE-packed weight whose product of the raw residual rows came as ``parts``
    (:func:`skinny_slabs`): their sum scaled by the rows' RMSNorm (``sq``: sums of squares), rounded and rotated, k and v in the cache, as
    :func:`skinny_gemm` with ``rope`` leaves them."""
    slices, t, n = parts.shape
    if not w.rope or n != w.n or parts.dtype != torch.float32 or not parts.is_contiguous() or slices not in (1, 2, 4, 8, 16):
        raise ValueError("parts must be skinny_slabs' of a RoPE-packed weight")
    if sq.dtype != torch.float32 or sq.numel() != t or not sq.is_contiguous():
        raise ValueError("sq must be a contiguous fp32 vector, one a row")
    cache = _rope_args(rope, t)
    qkv = torch.empty((t, n), dtype=torch.bfloat16, device=parts.device)
    rc = _lib.lib().kgs_rope_cache_packed_bf16(qkv.data_ptr(), rope["cos"].data_ptr(), rope["sin"].data_ptr(), rope["positions"].data_ptr(),
                                               rope["slots"].data_ptr(), cache.data_ptr(), t, *w.rope, n, parts.data_ptr(), slices, sq.data_ptr(),
                                               1.0 / w.k, float(eps), _lib.stream_handle(qkv.device))
    if rc:
        _lib.check(rc, "rope_cache_packed")
    return qkv


def _rope_args(rope: dict, m: int):
    """The cache of :func:`skinny_gemm`'s ``rope``, checked."""
    cache = rope["cache"]
    if cache.dtype != torch.bfloat16 or not cache.is_contiguous():
        raise ValueError("the RoPE epilogue writes a bf16 KV cache")
    for key in ("positions", "slots"):
        v = rope[key]
        if v.dtype != torch.int32 or not v.is_contiguous() or v.numel() < m:
            raise ValueError(f"{key} must be a contiguous int32 vector of >= M elements")
    return cache


def skinny_few(x: torch.Tensor, w: PackedWeight, out: torch.Tensor | None = None, norm: bool = False, resid: bool = False,
               eps: float = 1e-5, rope: dict | None = None) -> torch.Tensor:
    """:func:`skinny_gemm` of few rows (:func:`few_takes`), whose RMSNorm (``norm``; its weight folded into W) takes the rows'
    statistics from x itself; ``resid``: ``out += x @ W^T``. ``rope`` as there."""
    if x.dtype != torch.bfloat16 or not x.is_cuda or x.dim() != 2 or x.stride(1) != 1:
        raise ValueError("x must be a row-major bf16 GPU matrix")
    m, k = x.shape
    if k != w.k or not (few_takes(m, w.n, k, w.fp8, not norm and rope is None) or (not w.fp8 and few_wide(m, w.n, k))):
        raise ValueError(f"not a product of few rows: x {tuple(x.shape)}, W [{w.n}, {w.k}]")
    if (rope is not None) != bool(w.rope) or (resid and (rope is not None or w.swiglu)):
        raise ValueError("rope= needs a rope-packed qkv weight and vice versa; resid a plain one")
    if out is None:
        if resid:
            raise ValueError("resid needs the residual stream as out [M, N]")
        out = torch.empty((m, w.n_out), dtype=torch.bfloat16, device=x.device)
    elif out.dtype != torch.bfloat16 or tuple(out.shape) != (m, w.n_out) or out.stride(1) != 1 or out.device != x.device:
        raise ValueError("out must be a row-major bf16 matrix [M, N]")
    epi = (EPI_SWIGLU | GATE_EPI[w.act.act] if w.swiglu else 0) | (EPI_RMS if norm else 0) | (EPI_RESID if resid else 0)
    extra = (None,) * 5 + (0, 0)
    if rope is not None:
        cache = _rope_args(rope, m)
        epi |= EPI_ROPE
        extra = (rope["cos"].data_ptr(), rope["sin"].data_ptr(), rope["positions"].data_ptr(), rope["slots"].data_ptr(),
                 cache.data_ptr(), *w.rope)
    rc = _lib.lib().kgs_skinny_few(w.data.data_ptr(), x.data_ptr(), out.data_ptr(), m, w.n, k, x.stride(0), out.stride(0), epi,
                                   float(eps), w.act.limit, *extra, _lib.stream_handle(x.device))
    _lib.check(rc, f"skinny_few[{m}x{w.n}x{k}, epi={epi}]")
    return out


def skinny_few_two(x: torch.Tensor, w: PackedWeight, x2: torch.Tensor, w2: PackedWeight) -> tuple[torch.Tensor, torch.Tensor]:
    """Two plain products of :func:`skinny_few` of the same sizes and row strides in one launch."""
    m, k = x.shape
    for t, p in ((x, w), (x2, w2)):
        if t.dtype != torch.bfloat16 or not t.is_cuda or tuple(t.shape) != (m, p.k) or t.stride() != (x.stride(0), 1) or t.device != x.device:
            raise ValueError("x and x2 must be row-major bf16 GPU matrices of one shape and stride")
        if p.n != w.n or p.k != k or p.swiglu or p.rope or not few_takes(m, p.n, k, p.fp8, True):
            raise ValueError(f"not two products of few rows: x {tuple(t.shape)}, W [{p.n}, {p.k}]")
    out = torch.empty((2, m, w.n), dtype=torch.bfloat16, device=x.device)
    rc = _lib.lib().kgs_skinny_few_two(w.data.data_ptr(), x.data_ptr(), out[0].data_ptr(), w2.data.data_ptr(), x2.data_ptr(), out[1].data_ptr(),
                                       m, w.n, k, x.stride(0), w.n, _lib.stream_handle(x.device))
    _lib.check(rc, f"skinny_few_two[{m}x{w.n}x{k}]")
    return out[0], out[1]


def skinny_gemm(x: torch.Tensor, w: PackedWeight, out: torch.Tensor | None = None,
                ksplit: int | None = None, variant: int = 0, rms: torch.Tensor | None = None,
                resid_ss: torch.Tensor | None = None, zero: torch.Tensor | None = None,
                eps: float = 1e-5, rope: dict | None = None, counters: torch.Tensor | None = None, norm: bool = False,
                resid: bool = False) -> torch.Tensor:
    """``x @ W^T`` (bf16, fp32 accumulate) for ``x: [M <= 256, K]`` row-major;
    ``silu(x @ Wg^T) * (x @ Wu^T)`` for a ``swiglu`` weight. Fused epilogues:

    * ``rms`` (fp32 ``[M]`` row sums of squares of x): RMSNorm folded in -- the
      rows are scaled by ``rsqrt(rms / K + eps)`` (the norm weight must be folded
      into W, ``PackedWeight(..., fold=w)``);
    * ``resid_ss`` (fp32 ``[M]``): ``out`` is the residual stream, updated in
      place (``out += x @ W^T``), and the new rows' sums of squares are added
      into ``resid_ss`` (for the next ``rms`` consumer);
    * ``zero`` (fp32 ``[M]``): cleared at kernel start (a consumed statistic);
    * ``rms``, ``resid_ss`` and ``zero`` may be int64 ``[SUM_WORDS, M]`` instead (``resid_ss`` and ``zero`` alike,
      rows of at most ``SUM_MAX_N``): exact sums, whose bits do not depend on the order in which
      workgroups add to them;
    * ``rope`` (a ``rope=(H, HKV)``-packed qkv weight): dict of ``cos``, ``sin``
      (fp32 ``[max_pos, 64]``), ``positions`` and ``slots`` (int32 ``[M]``) and
      ``cache`` (the layer's bf16 pages): q / k rotated at their positions, k / v
      written into their cache slots -- :func:`rope_cache_` in the epilogue;
    * ``norm`` (instead of ``rms``; up to 64 rows of bf16 weights): RMSNorm folded in by statistics that the product
      makes from x itself; ``resid`` (instead of ``resid_ss``): the residual update alone;
    * ``counters`` (zeroed int32, a value per W strip; left zeroed): instead of the per-GPU ones, with
      slabs of the call's own -- calls that other streams' calls may overlap."""
    if x.dtype != torch.bfloat16 or not x.is_cuda or x.dim() != 2 or x.stride(1) != 1:
        raise ValueError("x must be a row-major bf16 GPU matrix")
    m, k = x.shape
    if k != w.k:
        raise ValueError(f"inner dims differ: x {tuple(x.shape)} vs W [{w.n}, {w.k}]")
    if w.fp8 and _mt(m) > 4:
        raise ValueError("fp8 (W8A16) skinny GEMM covers batches <= 64")
    if variant == 0 and ksplit is None:
        variant, ks = _skinny_plan(m, w.n, k, w.fp8, rope is not None)
    else:
        ks = ksplit if ksplit is not None else choose_ksplit(m, w.n, k, variant=variant)
    rps, kpc, mpad = skinny_geometry(m, variant)
    if w.n % rps or k % kpc:
        raise ValueError(f"skinny GEMM needs N % {rps} == 0 and K % {kpc} == 0 (N={w.n}, K={k})")
    if (norm and (rms is not None or resid or resid_ss is not None or w.fp8 or m > 64 or (ks > 1 and variant in KIN_VARIANTS))) or (resid and (resid_ss is not None or rope is not None)):
        raise ValueError("norm: a product of up to 64 rows of bf16 weights without rms or a residual update; resid: without resid_ss and rope")
    epi = (EPI_SWIGLU | GATE_EPI[w.act.act] if w.swiglu else 0) | (EPI_RMS if rms is not None else 0) | \
        (EPI_RMS | EPI_OWN if norm else 0) | (EPI_RESID if resid or resid_ss is not None else 0)
    for t, name, sums in ((rms, "rms", EPI_SUMS_IN), (resid_ss, "resid_ss", EPI_SUMS_OUT), (zero, "zero", EPI_SUMS_OUT)):
        if t is None:
            continue
        if t.dtype == torch.int64 and t.shape == (SUM_WORDS, m):
            epi |= sums
        elif t.dtype != torch.float32 or t.numel() < m:
            raise ValueError(f"{name} must be a contiguous fp32 vector of >= M elements, or int64 [{SUM_WORDS}, M]")
        if not t.is_contiguous():
            raise ValueError(f"{name} must be contiguous")
    if epi & EPI_SUMS_OUT and resid_ss is not None and zero is not None and resid_ss.dtype != zero.dtype:
        raise ValueError("resid_ss and zero must be of one kind")
    if epi & EPI_RESID:
        if w.swiglu or out is None or tuple(out.shape) != (m, w.n):
            raise ValueError("resid_ss needs the residual stream as out [M, N] (and no swiglu)")
    if out is None:
        out = torch.empty((m, w.n_out), dtype=torch.bfloat16, device=x.device)
    need = ks * mpad * (w.n + (2 * (w.n // rps) if norm else 0)) if ks > 1 else 0
    if counters is None:
        ws, cnt = _workspace(x.device, need, w.n // rps)
    else:
        if counters.dtype != torch.int32 or not counters.is_contiguous() or counters.numel() < w.n // rps:
            raise ValueError(f"counters must be at least {w.n // rps} contiguous int32")
        ws, cnt = torch.empty(need, dtype=torch.float32, device=x.device) if need else None, counters
    if (rope is not None) != bool(w.rope):
        raise ValueError("rope= needs a rope-packed qkv weight (PackedWeight(..., rope=(H, HKV))) and vice versa")
    if rope is not None:
        if w.fp8 or resid_ss is not None:
            raise ValueError("the RoPE epilogue is bf16-weight only and writes a fresh qkv output")
        cache = _rope_args(rope, m)
        rc = _lib.lib().kgs_skinny_gemm_bf16_rope(
            w.data.data_ptr(), x.data_ptr(), out.data_ptr(), None if ws is None else ws.data_ptr(), cnt.data_ptr(), m, w.n, k, x.stride(0),
            out.stride(0), ks, variant, epi & (EPI_RMS | EPI_SUMS_IN | EPI_OWN),
            rms.data_ptr() if rms is not None else None, 1.0 / k, float(eps), rope["cos"].data_ptr(),
            rope["sin"].data_ptr(), rope["positions"].data_ptr(), rope["slots"].data_ptr(), cache.data_ptr(),
            w.rope[0], w.rope[1], _lib.stream_handle(x.device))
        _lib.check(rc, f"skinny_gemm_rope[{m}x{w.n}x{k}, variant={variant}, ksplit={ks}]")
        return out
    rc = _lib.lib().kgs_skinny_gemm_bf16_fused(
        w.data.data_ptr(), x.data_ptr(), out.data_ptr(), None if ws is None else ws.data_ptr(), cnt.data_ptr(), m, w.n, k, x.stride(0),
        out.stride(0), ks, variant, epi, rms.data_ptr() if rms is not None else None,
        resid_ss.data_ptr() if resid_ss is not None else None, zero.data_ptr() if zero is not None else None,
        1.0 / k, float(eps), w.wscale.data_ptr() if w.fp8 else None, w.act.limit, _lib.stream_handle(x.device))
    _lib.check(rc, f"skinny_gemm[{m}x{w.n}x{k}, variant={variant}, ksplit={ks}, epi={epi}, fp8={w.fp8}]")
    return out


def reserve_workspace(device) -> None:
    """Allocate the largest split-K slab buffers the decode GEMMs can ask for up
    front (skinny: 64 MB; the 256x256 split-K kernel: SPLITK_WS_FLOATS), e.g.
    before hipGraph capture."""
    from .gemm import reserve_splitk_workspace

    _workspace(torch.device(device), 16 << 20, 1 << 16)
    reserve_splitk_workspace(torch.device(device), SPLITK_WS_FLOATS)


# ----------------------------------------------------------------------------
# paged KV cache

def kv_index_tables(device="cpu") -> tuple[torch.Tensor, torch.Tensor]:
    """``(K_IDX, V_IDX)``, each ``[32, 128]`` int64: the position of token ``tau``,
    dim ``d`` inside a page's K / V region (``kv_k_index`` / ``kv_v_index`` in
    decode.hip). K is in S^T = K.Q^T A-fragment order, V in O^T = V^T.P^T
    A-fragment order with the token order S^T's accumulator produces."""
    tau = torch.arange(PAGE, device=device)[:, None]
    d = torch.arange(HEAD_DIM, device=device)[None, :]
    k_idx = (((tau >> 4) * 4 + (d >> 5)) * 64 + ((d >> 3) & 3) * 16 + (tau & 15)) * 8 + (d & 7)
    v_idx = ((d >> 4) * 64 + ((tau >> 2) & 3) * 16 + (d & 15)) * 8 + (tau & 3) + 4 * (tau >> 4)
    return k_idx, v_idx


class PagedKVCache:
    """All layers' KV pages in one allocation: ``[layers, pages, kv_heads, 2, 4096]``
    (2 = K then V region of a 32-token page) in bf16, or in OCP e4m3
    (``dtype="fp8"``: scale 1, saturating -- half the bytes the decode attention
    streams and twice the tokens per GB). Pages are handed out by the
    scheduler's block allocator (kgs.serve)."""

    def __init__(self, layers: int, pages: int, kv_heads: int, device, dtype="bf16"):
        self.layers, self.pages, self.kv_heads = layers, pages, kv_heads
        tdt = {"bf16": torch.bfloat16, torch.bfloat16: torch.bfloat16, "fp8": FP8, FP8: FP8}[dtype]
        self.data = torch.zeros(layers, pages, kv_heads, 2, PAGE * HEAD_DIM, dtype=tdt, device=device)

    def layer(self, i: int) -> torch.Tensor:
        return self.data[i]

    @property
    def fp8(self) -> bool:
        return self.data.dtype == FP8

    @staticmethod
    def bytes_per_page(layers: int, kv_heads: int, dtype="bf16") -> int:
        return layers * kv_heads * 2 * PAGE * HEAD_DIM * (1 if dtype == "fp8" else 2)


def rope_cache_(qkv: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, positions: torch.Tensor,
                slots: torch.Tensor, cache_layer: torch.Tensor, heads: int, kv_heads: int,
                partials: torch.Tensor | None = None, rows: torch.Tensor | None = None) -> torch.Tensor:
    """In place: rotate the q and k heads of every row of the fused ``qkv``
    ``[T, (H + 2 HKV) * 128]`` at ``positions[t]``, and write k, v into cache slot
    ``slots[t]`` (``page * 32 + offset``; < 0 skips the write).

    ``partials`` (fp32 ``[nslice, T, (H + 2 HKV) * 128]``, from
    ``kgs.ops.gemm.gemm_nt_w4x_partials``): the projection arrives as split-K
    partial products; they are reduced (bf16-rounded like the unfused reduce)
    in the same launch and ``qkv`` is output only.

    ``rows`` (int32, one per token): token ``t`` is row ``rows[t]`` of ``qkv``, none where negative --
    prompts padded to whole pages whose padding has no rows."""
    t = qkv.shape[0]
    if rows is not None:
        t = rows.numel()
        if rows.dtype != torch.int32 or not rows.is_contiguous():
            raise ValueError("rows must be a contiguous int32 vector")
    if qkv.dtype != torch.bfloat16 or not qkv.is_cuda or qkv.stride(1) != 1:
        raise ValueError("qkv must be a row-major bf16 GPU matrix")
    nslice = 0
    if partials is not None:
        if partials.dtype != torch.float32 or partials.dim() != 3 or not partials.is_contiguous() or \
                tuple(partials.shape[1:]) != (qkv.shape[0], (heads + 2 * kv_heads) * HEAD_DIM):
            raise ValueError("partials must be contiguous fp32 [nslice, rows of qkv, (H + 2 HKV) * 128]")
        nslice = partials.shape[0]
    for v, name in ((positions, "positions"), (slots, "slots")):
        if v.dtype != torch.int32 or not v.is_contiguous() or v.numel() != t:
            raise ValueError(f"{name} must be a contiguous int32 vector of length {t}")
    for v in (cos, sin):
        if v.dtype != torch.float32 or not v.is_contiguous() or v.shape[-1] != HEAD_DIM // 2:
            raise ValueError("cos/sin must be contiguous fp32 [max_pos, 64]")
    if cache_layer.dtype not in (torch.bfloat16, FP8) or not cache_layer.is_contiguous():
        raise ValueError("cache_layer must be a contiguous bf16 or e4m3 page array")
    rc = _lib.lib().kgs_rope_cache_bf16(qkv.data_ptr(), cos.data_ptr(), sin.data_ptr(), positions.data_ptr(),
                                        slots.data_ptr(), cache_layer.data_ptr(), t, heads, kv_heads, HEAD_DIM,
                                        qkv.stride(0), 1 if cache_layer.dtype == FP8 else 0,
                                        None if partials is None else partials.data_ptr(), nslice,
                                        None if rows is None else rows.data_ptr(), qkv.shape[0],
                                        _lib.stream_handle(qkv.device))
    _lib.check(rc, "rope_cache")
    return qkv


def decode_splits(batch: int, kv_heads: int, max_pages: int, cus: int = CUS, min_pages: int = 4) -> tuple[int, int]:
    """(pages_per_split, nsplit) for a block-table width of ``max_pages``.

    Split each context so that the grid holds about two waves per CU:
    ``nsplit = ceil(2 * CUs / (batch * kv_heads))``. Every split keeps at least
    ``min_pages`` pages (a one-page split is all launch and merge overhead: 52
    us for batch 1 x 4096 tokens with 1-page splits, profiles/decode_kernels.md).
    So batch 1-8 takes eight splits, batch 16 four and batch 32 two. From batch
    64 up, one split per (sequence, KV head) is fastest. It is paired with the
    two-page register pipeline, which the kernel runs for grids of up to 1024
    waves (``kgs_paged_decode_bf16``).

    Round-3 measurements (``profiles/r3/decode/paged_sweep_ctx*.log``, table
    width 64 pages):

    * 1024 cached tokens: batch 64 52 us (was 100 with the old rule of two
      splits and no pipeline); batch 128 92 us (was 124);
    * 528 tokens: batch 64 30 us (was 59), batch 128 50 us (was 72);
    * 2000 tokens: within 2 % of the best split everywhere.

    The old rule split large batches whenever the table held 64 pages or more;
    without the pipeline, each split paid one page latency per page."""
    groups = max(1, batch * kv_heads)
    want = max(1, math.ceil(2 * cus / groups))
    nsplit = max(1, min(math.ceil(max_pages / min_pages), want))
    pps = math.ceil(max_pages / nsplit)
    return pps, math.ceil(max_pages / pps)


def workgroup_splits(batch: int, kv_heads: int, max_pages: int, cus: int = CUS) -> int:
    """Parts of every sequence's pages for the attention by workgroups. Two workgroups per
    CU read the cache fastest, so parts are made up to there: of at least 8 pages by the table's
    width while most CUs idle, of 32 from half the CUs on, where a merge costs as much as
    the shorter parts save (us, 8 KV heads: one sequence of 4000 tokens 42 / 16 / 11 in 1 / 4 / 16
    parts; 16 of 1000 15.0 / 17.2 in 1 / 4; 16 unequal ones of up to 4000 27.7 / 22.3)."""
    groups = batch * kv_heads
    return min(-(-2 * cus // groups), max(1, max_pages // (8 if 2 * groups < cus else 32)))


def shorter_parts(batch: int, kv_heads: int, max_pages: int, waves: int, fp8: bool) -> tuple[int, int]:
    """(parts, waves) of that attention in equal parts: :func:`workgroup_splits`, but few pairs in narrow tables are one chain of page latencies, which parts of four pages by
    four waves shorten by more than their merge costs. us before / so: 8 KV heads in 16 pages 1 / 4 sequences of 500 tokens 7.9, 8.7 / 6.7, 7.5, 4 of up to 500 8.1 / 7.1,
    one of 260 6.6 / 6.3, e4m3 1 / 4 of 500 7.5, 8.1 / 6.7, 7.6; in 32 pages one of 1000 8.2 / 7.5, of 520 7.1 / 7.0, with 4 KV heads 8.0, 6.9 / 7.3, 6.8; not 4 sequences of
    1000 there, 9.2 / 9.6, nor e4m3, 7.9 / 8.0. A step of four layers, contexts of 300 in 16 pages: 2048 wide with 4 KV heads 1, 2, 4, 8 sequences 172, 176, 179, 189 / 170, 171,
    176, 186; 4096 wide with 8 361, 364, 368 / 358, 364, 366 of 1, 2, 4; not 64 pairs, 378 / 381."""
    n, pairs = workgroup_splits(batch, kv_heads, max_pages), batch * kv_heads
    least = 4 if 16 <= max_pages < 32 and pairs <= 32 else 8 if 32 <= max_pages < 64 and pairs <= 8 and not fp8 else 1
    return (least, min(waves, 4)) if n < least else (n, waves)


def workgroup_waves(groups: int, max_pages: int, fp8: bool) -> int:
    """Waves of such a workgroup for ``groups`` (sequence, KV head) pairs, 1 for the kernel of single waves.

    Eight (e4m3 pages four), except where the table is so narrow that a wave has a page or two: a workgroup's fixed
    cost counts then, more so the more pairs a CU has. At 32 pages the waves of one group even out unequal contexts
    for more than they cost. us with 8 KV heads, contexts as long as the table / uniform up to there:

    ======  =========  =====  ==============  ===============  =====================
    pages    sequences  type  single waves    8 (e4m3: 4)      this rule (waves)
    ======  =========  =====  ==============  ===============  =====================
    1        32         bf16  3.5             3.8              3.5 (1)
    1        100        bf16  3.9             6.3              3.9 (1)
    2        256        bf16  11.7 / 9.5      17.3 / 16.1      11.7 / 9.5 (1)
    4        100        bf16  9.7 / 7.0       10.6 / 8.3       8.9 / 6.3 (4)
    4        256        bf16  22.0 / 16.7     24.5 / 19.0      21.6 / 14.7 (2)
    8        1024       bf16  170 / 110       171 / 104        173 / 102 (4)
    32       256        bf16  156 / 113       163 / 90         163 / 90 (8)
    2        100        e4m3  5.4 / 6.1       6.7 / 6.6        4.8 / 5.0 (2)
    2        130        e4m3  6.1 / 6.0       8.7 / 8.5        6.1 / 6.0 (1)
    2        1024       e4m3  26 / 22         55 / 52          26 / 22 (1)
    4        160        e4m3  9.8 / 9.4       11.8 / 11.1      9.8 / 9.4 (1)
    8        181        e4m3  19.9 / 16.1     19.7 / 16.0      20.3 / 14.5 (2)
    8        256        e4m3  23.3 / 17.9     26.9 / 21.1      23.3 / 17.9 (1)
    16       256        e4m3  44.6 / 30.6     43.8 / 31.3      45.3 / 27.5 (2)
    32       256        e4m3  84.8 / 58.5     81.1 / 50.6      81.1 / 50.6 (4)
    ======  =========  =====  ==============  ===============  =====================
    """
    if fp8:
        if groups < 640:
            return 4
        if max_pages <= (8 if groups >= 1536 else 4 if groups >= 1152 else 2 if groups >= 1024 else 1):
            return 1
        return 2 if max_pages <= 16 else 4
    if max_pages <= (2 if groups >= 2048 else 1):
        return 1
    if max_pages <= 4 and groups >= 1024:
        return 2
    return 4 if max_pages <= 8 else 8


PARTS_LEAST = 8  # pages of such a part at least


def length_parts(batch: int, kv_heads: int, max_pages: int, waves: int, fp8: bool) -> int:
    """Parts that the pages are dealt to where they follow the sequences' lengths, 0 for equal parts of each.

    For 3 to 128 sequences and tables of 64 pages on: up to two have equal parts that are as good (one of 4000 tokens 10.2 us /
    10.6), narrower tables hold lengths that differ by less than the longer start costs (256 sequences of 32 pages
    26.6 / 28.0), and 256 sequences of 600 on average, four rounds of workgroups that even out by themselves, take 47.9 /
    49.4. One and a half workgroups per CU, and fewer than one up to three fifths of the CUs in (sequence, KV head) pairs, whose short last
    parts come on top. us, equal parts / 192 workgroups / 384, lengths log-normal around the mean: 24 of 3676 tokens with 8 KV heads
    67.9 / 70.4 / 58.8, 27 of 2222 44.5 / 46.2 / 40.3, 51 of 1826 with 4 44.9 / 48.4 / 40.4, 100 of 700 38.1 / 30.8 / 29.9; 16 of 1000 with 8 17.9 / 17.1 /
    18.3, 8 of 2348 19.3 / 18.4 / 21.0. Over 380 batches the geometric mean is 0.75 to 0.92 of the equal parts' time by the number of pairs. Slower are
    short contexts in tables that are much wider (101 of 117 tokens in 256 pages 6.5 / 7.7), equal ones that just need a second part (72 of
    605 in a batch of 128 21.2 / 27.3) and 128 of up to 2000, uniform,
    with 4 KV heads (53.2 / 54.7)."""
    if max_pages < 64 or not 2 < batch <= 128 or waves != (4 if fp8 else 8):
        return 0
    return max(1, (192 if 5 * batch * kv_heads < 3 * CUS else 384) // kv_heads)


def part_target(batch: int, kv_heads: int, max_pages: int, waves: int, fp8: bool) -> int:
    """:func:`length_parts`, 0 where equal parts are as short: up to 40 pairs and tables of fewer than 128 pages, 8 pages a part at most
    (us, equal / by length: 5 of 747 tokens with 4 KV heads 9.6 / 11.4, 3 of 2138 with 8 11.0 / 12.1, 14 of 3173 with 1 12.7 / 14.0; 11 of 1132 with 4,
    44 pairs, 12.9 / 12.1, and 5 of 3098 in 128 pages 15.1 / 13.8)."""
    return 0 if batch * kv_heads <= 40 and max_pages < 128 else length_parts(batch, kv_heads, max_pages, waves, fp8)


def part_tickets(batch: int, kv_heads: int, max_pages: int, fp8: bool) -> int:
    """Length of the ``tickets`` that :func:`paged_decode_attention` of such a batch takes, 0: none."""
    waves = workgroup_waves(batch * kv_heads, max_pages, fp8)
    return batch * kv_heads if part_target(batch, kv_heads, max_pages, waves, fp8) else 0


_AWS: dict = {}


def _attn_workspace(b: int, heads: int, kv_heads: int, nsplit: int, device) -> tuple:
    """(po, pml, cnt) split-merge workspace of the paged decode attention
    (None x 3 for one split); grown on demand, one per device: calls that share it are ordered by their stream."""
    if nsplit <= 1:
        return None, None, None
    need = b * heads * nsplit
    key = device_key(device)
    po, pml, cnt = _AWS.get(key, (None, None, None))
    if po is None or po.numel() < need * HEAD_DIM or cnt.numel() < b * kv_heads:
        retire(po, pml, cnt)
        po = torch.empty(max(need, 1 << 14) * HEAD_DIM, dtype=torch.float32, device=device)
        pml = torch.empty(max(need, 1 << 14) * 2, dtype=torch.float32, device=device)
        cnt = torch.zeros(max(b * kv_heads, 4096), dtype=torch.int32, device=device)
        _AWS[key] = (po, pml, cnt)
    return po, pml, cnt


def rope_paged_decode_attention(partials: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                                positions: torch.Tensor, slots: torch.Tensor, cache_layer: torch.Tensor,
                                block_tables: torch.Tensor, ctx_lens: torch.Tensor, heads: int, kv_heads: int,
                                out: torch.Tensor | None = None, scale: float | None = None,
                                pages_per_split: int | None = None, pipe: bool | None = None) -> torch.Tensor:
    """:func:`rope_cache_` (partials form) and :func:`paged_decode_attention` in
    ONE launch (``kgs_paged_decode_rope_bf16``): ``partials`` fp32
    ``[nslice, B, (H + 2 HKV) * 128]`` from ``gemm_nt_w4x_partials`` of the
    fused qkv projection. Each attention wave reduces, rotates and caches its
    own (sequence, KV head) rows, so the rotated q never goes through memory
    and the rope_cache launch disappears. Same cache contents and output as the
    two launches. ``slots[b]`` must lie in the last page of ``ctx_lens[b]``
    (the engine's assignment)."""
    nh = heads + 2 * kv_heads
    if partials.dtype != torch.float32 or partials.dim() != 3 or not partials.is_contiguous() or \
            partials.shape[2] != nh * HEAD_DIM or not partials.is_cuda:
        raise ValueError("partials must be contiguous fp32 GPU [nslice, B, (H + 2 HKV) * 128]")
    b = partials.shape[1]
    if partials.shape[0] not in (2, 4, 8):
        raise ValueError("rope_paged_decode_attention: 2, 4 or 8 K slices (compile-time in the kernel)")
    if heads % kv_heads or heads // kv_heads > 6:
        raise ValueError("rope_paged_decode_attention: GQA group of at most 6 q heads per KV head")
    for v, name in ((positions, "positions"), (slots, "slots"), (ctx_lens, "ctx_lens")):
        if v.dtype != torch.int32 or not v.is_contiguous() or v.numel() != b:
            raise ValueError(f"{name} must be a contiguous int32 vector of length {b}")
    for v in (cos, sin):
        if v.dtype != torch.float32 or not v.is_contiguous() or v.shape[-1] != HEAD_DIM // 2:
            raise ValueError("cos/sin must be contiguous fp32 [max_pos, 64]")
    if cache_layer.dtype not in (torch.bfloat16, FP8) or not cache_layer.is_contiguous():
        raise ValueError("cache_layer must be a contiguous bf16 or e4m3 page array")
    if block_tables.dtype != torch.int32 or not block_tables.is_contiguous() or block_tables.shape[0] != b:
        raise ValueError("block_tables must be contiguous int32 [B, max_pages]")
    max_pages = block_tables.shape[1]
    if pages_per_split is None:
        pps, nsplit = decode_splits(b, kv_heads, max_pages)
    else:
        pps, nsplit = pages_per_split, math.ceil(max_pages / pages_per_split)
    if out is None:
        out = torch.empty((b, heads * HEAD_DIM), dtype=torch.bfloat16, device=partials.device)
    po, pml, cnt = _attn_workspace(b, heads, kv_heads, nsplit, partials.device)
    scale = 1.0 / math.sqrt(HEAD_DIM) if scale is None else scale
    rc = _lib.lib().kgs_paged_decode_rope_bf16(
        partials.data_ptr(), partials.shape[0], cos.data_ptr(), sin.data_ptr(), positions.data_ptr(),
        slots.data_ptr(), cache_layer.data_ptr(), block_tables.data_ptr(), ctx_lens.data_ptr(), out.data_ptr(),
        po.data_ptr() if po is not None else None, pml.data_ptr() if pml is not None else None,
        cnt.data_ptr() if cnt is not None else None, b, heads, kv_heads, HEAD_DIM, max_pages, pps, nsplit,
        out.stride(0), float(scale), 1 if cache_layer.dtype == FP8 else 0, -1 if pipe is None else int(bool(pipe)),
        _lib.stream_handle(partials.device))
    _lib.check(rc, "rope_paged_decode_attention")
    return out


def paged_decode_attention(q: torch.Tensor, cache_layer: torch.Tensor, block_tables: torch.Tensor,
                           ctx_lens: torch.Tensor, heads: int, kv_heads: int, out: torch.Tensor | None = None,
                           scale: float | None = None, pages_per_split: int | None = None,
                           pipe: bool | None = None, tickets: torch.Tensor | None = None) -> torch.Tensor:
    """One query token per sequence: ``q`` rows ``[B, >= H*128]`` (e.g. the rotated
    q heads at the front of the fused QKV rows), ``block_tables`` int32
    ``[B, max_pages]``, ``ctx_lens`` int32 ``[B]`` (cached tokens incl. the new
    one). Returns ``[B, H*128]`` bf16. Parts that follow the lengths (:func:`part_target`) have partial results of the call's own and take
    ``tickets``, zeroed int32 of :func:`part_tickets` values or more, which are zero again behind it and so serve every layer of
    a step (None: the call's own, a launch of 1.5 us more). Contexts split in any other way
    share one workspace per GPU: calls of such batches on several streams have to be ordered."""
    b = q.shape[0]
    if q.dtype != torch.bfloat16 or not q.is_cuda or q.stride(1) != 1:
        raise ValueError("q must be a row-major bf16 GPU matrix")
    if block_tables.dtype != torch.int32 or not block_tables.is_contiguous() or block_tables.shape[0] != b:
        raise ValueError("block_tables must be contiguous int32 [B, max_pages]")
    if ctx_lens.dtype != torch.int32 or not ctx_lens.is_contiguous() or ctx_lens.numel() != b:
        raise ValueError("ctx_lens must be contiguous int32 [B]")
    max_pages = block_tables.shape[1]
    fp8 = cache_layer.dtype == FP8
    waves = workgroup_waves(b * kv_heads, max_pages, fp8) if pages_per_split is None and pipe is None else 1
    target = part_target(b, kv_heads, max_pages, waves, fp8)
    if waves > 1:
        nsplit, waves = shorter_parts(b, kv_heads, max_pages, waves, fp8) if b else (1, waves)
    elif pages_per_split is None:
        pps, nsplit = decode_splits(b, kv_heads, max_pages)
    else:
        pps, nsplit = pages_per_split, math.ceil(max_pages / pages_per_split)
    if out is None:
        out = torch.empty((b, heads * HEAD_DIM), dtype=torch.bfloat16, device=q.device)
    scale = 1.0 / math.sqrt(HEAD_DIM) if scale is None else scale
    if target:
        rows = (b + target) * heads  # of partial results, then their maxima and sums
        part = torch.empty(rows * (HEAD_DIM + 2), dtype=torch.float32, device=q.device)
        if tickets is None:
            tickets = torch.zeros(b * kv_heads, dtype=torch.int32, device=q.device)
        elif tickets.dtype != torch.int32 or tickets.device != q.device or not tickets.is_contiguous() or tickets.numel() < b * kv_heads:
            raise ValueError(f"tickets must be {b * kv_heads} contiguous int32 or more on q's GPU")
        rc = _lib.lib().kgs_paged_decode_wg_bal(q.data_ptr(), cache_layer.data_ptr(), block_tables.data_ptr(), ctx_lens.data_ptr(),
                                                out.data_ptr(), part.data_ptr(), part.data_ptr() + rows * HEAD_DIM * 4,
                                                tickets.data_ptr(), b, heads, kv_heads, HEAD_DIM, max_pages, target, PARTS_LEAST,
                                                q.stride(0), out.stride(0), float(scale), int(fp8), _lib.stream_handle(q.device))
        _lib.check(rc, "paged_decode_attention")
        return out
    po, pml, cnt = _attn_workspace(b, heads, kv_heads, nsplit, q.device)
    if waves > 1:
        rc = _lib.lib().kgs_paged_decode_wg_ex(q.data_ptr(), cache_layer.data_ptr(), block_tables.data_ptr(), ctx_lens.data_ptr(),
                                               out.data_ptr(), po.data_ptr() if po is not None else None,
                                               pml.data_ptr() if pml is not None else None,
                                               cnt.data_ptr() if cnt is not None else None, b, heads, kv_heads, HEAD_DIM,
                                               max_pages, nsplit, q.stride(0), out.stride(0), float(scale),
                                                  int(fp8), waves, _lib.stream_handle(q.device))
        _lib.check(rc, "paged_decode_attention")
        return out
    rc = _lib.lib().kgs_paged_decode_bf16_ex(q.data_ptr(), cache_layer.data_ptr(), block_tables.data_ptr(),
                                             ctx_lens.data_ptr(), out.data_ptr(),
                                             po.data_ptr() if po is not None else None,
                                             pml.data_ptr() if pml is not None else None,
                                             cnt.data_ptr() if cnt is not None else None, b, heads, kv_heads, HEAD_DIM,
                                             max_pages, pps, nsplit, q.stride(0), out.stride(0), float(scale),
                                             1 if cache_layer.dtype == FP8 else 0,
                                             -1 if pipe is None else int(bool(pipe)), _lib.stream_handle(q.device))
    _lib.check(rc, "paged_decode_attention")
    return out


# ----------------------------------------------------------------------------
# plain-PyTorch references (fp32 math; CPU or GPU)

def ref_cache_write(cache_layer: torch.Tensor, k: torch.Tensor, v: torch.Tensor, slots: torch.Tensor) -> None:
    """Scatter ``k, v: [T, HKV, 128]`` into ``cache_layer [pages, HKV, 2, 4096]``."""
    k_idx, v_idx = kv_index_tables(cache_layer.device)
    keep = slots >= 0
    slots = slots[keep].long()
    k, v = k[keep], v[keep]
    page, tau = slots // PAGE, slots % PAGE
    hkv = cache_layer.shape[1]

    def cvt(t):
        if cache_layer.dtype == FP8:  # saturating, like the kernel
            return t.float().clamp(-FP8_MAX, FP8_MAX).to(FP8)
        return t.to(cache_layer.dtype)

    for h in range(hkv):
        cache_layer[page[:, None], h, 0, k_idx[tau]] = cvt(k[:, h])
        cache_layer[page[:, None], h, 1, v_idx[tau]] = cvt(v[:, h])


def gather_kv_into(cache_layer: torch.Tensor, pages: torch.Tensor, ctx: int, k: torch.Tensor, v: torch.Tensor) -> None:
    """:func:`gather_kv` into the given row-major bf16 ``k``, ``v`` (of one row stride), in one
    launch; rows of a page outside the cache come back zero."""
    rows, hkv = k.shape[0], cache_layer.shape[1]
    if cache_layer.dtype not in (torch.bfloat16, FP8) or not cache_layer.is_contiguous():
        raise ValueError("the cache must be contiguous bf16 or e4m3")
    if pages.numel() < (ctx + PAGE - 1) // PAGE or not 0 <= ctx <= rows:
        raise ValueError(f"{pages.numel()} pages and {rows} rows for {ctx} tokens")
    if k.dtype != torch.bfloat16 or v.dtype != torch.bfloat16 or k.shape != v.shape or k.stride() != v.stride() or \
            k.shape[1] != hkv * HEAD_DIM or k.stride(1) != 1:
        raise ValueError("k and v must be row-major bf16 [rows, kv_heads * 128] of one row stride")
    pages = pages.to(cache_layer.device, torch.int32).contiguous()
    rc = _lib.lib().kgs_gather_kv(cache_layer.data_ptr(), pages.data_ptr(), k.data_ptr(), v.data_ptr(), ctx, rows, hkv, HEAD_DIM,
                                  cache_layer.shape[0], k.stride(0), 1 if cache_layer.dtype == FP8 else 0,
                                  _lib.stream_handle(k.device))
    _lib.check(rc, "gather_kv")


_KV_IDX: dict = {}


def gather_kv(cache_layer: torch.Tensor, pages: torch.Tensor, ctx: int, rows: int | None = None
              ) -> tuple[torch.Tensor, torch.Tensor]:
    """The first ``ctx`` cached tokens of one sequence as contiguous row-major
    ``k``, ``v`` ``[rows, kv_heads * 128]`` bf16 (rows ``ctx .. rows-1`` zero) --
    the keys/values a prefill chunk attends to (``rows`` pads them to the
    chunk's q-blocks). Vectorised torch gathers through the page layout's index
    tables; an fp8 cache is widened to bf16. :func:`gather_kv_into` is the one-launch form."""
    rows = ctx if rows is None else rows
    dev = cache_layer.device
    key = (dev.type, dev.index)
    if key not in _KV_IDX:
        _KV_IDX[key] = kv_index_tables(dev)
    k_idx, v_idx = _KV_IDX[key]
    hkv = cache_layer.shape[1]
    npg = (ctx + PAGE - 1) // PAGE
    sel = cache_layer[pages[:npg].long()]  # [npg, hkv, 2, 4096]
    out = []
    for region, idx in ((0, k_idx), (1, v_idx)):
        t = sel[:, :, region][..., idx]  # [npg, hkv, 32, 128]
        t = t.permute(0, 2, 1, 3).reshape(npg * PAGE, hkv * HEAD_DIM)[:ctx].to(torch.bfloat16)
        if rows > ctx:
            t = torch.cat([t, t.new_zeros(rows - ctx, hkv * HEAD_DIM)])
        out.append(t.contiguous())
    return out[0], out[1]


def ref_gather_kv(cache_layer: torch.Tensor, pages: torch.Tensor, ctx: int) -> tuple[torch.Tensor, torch.Tensor]:
    """The first ``ctx`` tokens of one sequence: ``(k, v)``, each ``[ctx, HKV, 128]`` fp32."""
    k_idx, v_idx = kv_index_tables(cache_layer.device)
    pos = torch.arange(ctx, device=cache_layer.device)
    page = pages.long()[pos // PAGE]
    tau = pos % PAGE
    hkv = cache_layer.shape[1]
    k = torch.stack([cache_layer[page[:, None], h, 0, k_idx[tau]] for h in range(hkv)], dim=1)
    v = torch.stack([cache_layer[page[:, None], h, 1, v_idx[tau]] for h in range(hkv)], dim=1)
    return k.float(), v.float()


def ref_paged_decode(q: torch.Tensor, cache_layer: torch.Tensor, block_tables: torch.Tensor, ctx_lens: torch.Tensor,
                     heads: int, kv_heads: int, scale: float | None = None) -> torch.Tensor:
    scale = 1.0 / math.sqrt(HEAD_DIM) if scale is None else scale
    rep = heads // kv_heads
    outs = []
    for i in range(q.shape[0]):
        ctx = int(ctx_lens[i])
        k, v = ref_gather_kv(cache_layer, block_tables[i], ctx)
        qi = q[i, :heads * HEAD_DIM].float().reshape(heads, HEAD_DIM)
        kk = k.repeat_interleave(rep, dim=1)  # [ctx, H, D]
        vv = v.repeat_interleave(rep, dim=1)
        s = torch.einsum("hd,thd->ht", qi, kk) * scale
        p = torch.softmax(s, dim=-1)
        outs.append(torch.einsum("ht,thd->hd", p, vv).reshape(-1))
    return torch.stack(outs)


def ref_rope_rows(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, positions: torch.Tensor,
                  heads: int) -> torch.Tensor:
    """Rotate-half RoPE of the first ``heads`` 128-wide heads of each row (fp32 result)."""
    t = x.shape[0]
    xf = x[:, :heads * HEAD_DIM].float().reshape(t, heads, HEAD_DIM)
    c, s = cos[positions.long()][:, None, :], sin[positions.long()][:, None, :]
    x1, x2 = xf[..., :HEAD_DIM // 2], xf[..., HEAD_DIM // 2:]
    return torch.cat((x1 * c - x2 * s, x2 * c + x1 * s), dim=-1).reshape(t, heads * HEAD_DIM)
