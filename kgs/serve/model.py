"""Paged-KV Llama model runner for :mod:`kgs.serve` (BASELINE config 5 stand-in:
Llama-3-8B bf16, TP=1, one MI355X).

Two step kinds, both driven by the native scheduler's plans
(``native/serve/scheduler.cpp``):

* **prefill** -- the prompts of newly admitted sequences, each padded to a
  multiple of 128 tokens and concatenated (the layers drop the padding where that
  saves a tile of rows; steps of up to ``fused_max_batch`` rows, 64 at most, run the FUSED layer
  below, of up to 128 the one IN SLICES where it pays, of up to 256 the split tiles): every projection is one
  :func:`kgs.ops.gemm_nt` (256x256 MFMA pipeline), RoPE + the KV-cache scatter
  is one :func:`kgs.ops.decode.rope_cache_` launch, attention is one
  flash-attention launch over all sequences' query blocks, and only the last real token of each
  sequence goes through the LM head;
* **decode** -- one token per running sequence; attention is
  :func:`kgs.ops.decode.paged_decode_attention` over the paged cache. Batches up
  to ``fused_max_batch`` run the FUSED layer: five
  :func:`kgs.ops.decode.skinny_gemm` launches over prepacked weights whose
  epilogues carry the RMSNorms (norm weights folded into the weights, row
  scales from sums of squares that the GEMMs make of their own input, or where
  they cannot the residual-updating ones accumulate), the residual adds and
  SwiGLU -- no elementwise kernels. From 33 to 128 rows (:meth:`ServingModel._slabs_pay`, :meth:`ServingModel._wide`; a
  ``fused_max_batch`` of 32 and less turns them off) the layer runs IN SLICES: products
  over the prepacked weights leave their K slices to the rotation and the residual adds that
  follow. Larger batches run
  split-K four-wave tiles (:func:`kgs.ops.decode.w4x_route`, :func:`kgs.ops.decode.w4x_rule`)
  whose partial sums go into the rotation, norm or gate that follows, and
  otherwise add_rmsnorm/silu_mul and hipBLASLt, the split-K 256x256 GEMM
  (:func:`kgs.ops.decode.splitk_slices`), the skinny GEMM
  (:func:`kgs.ops.decode.use_skinny`) or the 256x256 GEMM (LM head) where
  those measured faster.

``decode_weights="fp8"``: the decode copies are weight-only fp8 (W8A16, one
scale per output row, dequantised in registers), halving the weight bytes a
decode step streams; prefill and batches above the fused path stay bf16.

``kv_cache_dtype="fp8"``: e4m3 KV pages (scale 1), dequantised in the decode
attention's registers -- half the KV bytes per decode step.

``backend="ref"`` runs the same weights, cache layout and plans through plain
PyTorch (CPU or GPU) -- the numerics reference for tests.

Weights are random-init (no network, no checkpoint) with the same generator
scheme as :class:`kgs.models.llama.LlamaModel`, whose ``forward`` (no cache) is
the full-recompute oracle the tests compare generations against.
"""
from __future__ import annotations

import os

import torch

from kgs.models.llama import LlamaConfig, LlamaModel, _rms_norm
from kgs.ops import decode as D

from .trace import TRACE as T

GATE = 32  # outputs of the gate kernel's tiles: a route's width


def gate_up_panel_widths(n: int, k: int) -> set:
    """Tile widths of the unsplit SwiGLU decode routes for a gate|up of shape
    (n, k) (kgs.ops.decode.W4X_TUNED): one tile-panel copy is made per width."""
    return {r[0] for (_, rn, rk), r in D.W4X_TUNED.items() if (rn, rk) == (n, k) and r[1] == 1}


def gate_up_route(m: int, n: int, k: int):
    """The route of :meth:`ServingModel._swiglu_route` for a gate|up ``[n, k]`` without measured entries, None: the library and the product.

    The gate kernel by :func:`kgs.ops.decode.gate_rule`, beside the library's product as beside slices: 2048x3328 at 39 rows 10.6 us by the
    library, 16.3 by the gate kernel, 2048x6912 at 104 21.6 / 30.5. Where unsplit tiles take more rows of W than CUs have 64 of, only up to 40 rows
    and K of 4096 (33 rows of 25856x1536 19.8 / 19.3; 40 of 22528x8064 76 / 82, 56 of 23808x3840 43.5 / 47.5, 60 of 22272x7680 79 / 90). Over 170
    sizes of 1 to 128 rows its geometric mean is 0.67 of the other route's time, the worst 1.07 (32 of 21504x6912 62.6 / 67.0)."""
    rule = D.w4x_rule(m, n, k)
    whole = rule is not None and rule[1] == 1
    if whole and n > 64 * D.CUS and (m > 40 or k > 4096):
        return rule
    bm = D.gate_rule(m, n, k, sliced=not whole)
    return rule if bm is None else (GATE, 1, bm)


def head_on_small_tiles(m: int, n: int, k: int) -> bool:
    """Whether ``m`` rows of an LM head ``[n, k]`` go by the general kernel's small tiles and not by the library.

    Up to 32 rows of large vocabularies, which they read once and past the caches. us, library / so, 1 row: 32000x4096 58 / 47, 16384x2048
    18 / 16, 128256x2048 119 / 83; 32 rows 32000x2048 35 / 30, 64000x4096 118 / 90. Not below 16384 (1 row of 8192x4096 16.7 / 18.8, 12288x8192 40.6 / 43.6,
    5000x8192 19.9 / 23.4), nor where the rows' products are no longer hidden by the reads and the library has larger tiles that
    fit (32 rows of 18432x3072 28.7 / 33.4, 16 of 50432x5120 90.8 / 96.5, 32 of 50257x1024, whose outputs are not aligned, 23.5 /
    26.2). Worst within the rule: 1 row of 20480x8192 67.7 / 71.3, 32 of 18432x2048 22.1 / 22.8."""
    return 0 < m <= 32 and n >= 16384 and n % 8 == 0 and (k <= 2048 or k % 4096 == 0 or (m <= 16 and k <= 4096))


class _PromptRows:
    """Rows of a step's layers: ``n`` of them, ``last`` (int32) those whose logits are wanted, attention
    ``items`` (and ``merges``, ``slots`` of their parts) with the gathered contexts ``past`` ``(first row, end, tokens, portion)``, and, where
    the padding was dropped, ``keep`` (int32: the given rows that stay) and ``rows`` (int32: each
    given row's number, -1 for padding)."""

    __slots__ = ("n", "past", "items", "merges", "slots", "last", "rows", "keep")

    def __init__(self, n, past):
        self.n, self.past, self.slots = n, past, 0
        self.items = self.merges = self.last = self.rows = self.keep = None


class ServingModel:
    ragged = False      # prompt steps come padded, portions are multiples of pad_multiple
    pad_multiple = 128  # the flash-attention prefill kernel's q-block
    has_state = False   # no per-sequence recurrent state

    @classmethod
    def for_engine(cls, cfg: LlamaConfig, ec, device, backend: str, num_pages: int) -> "ServingModel":
        if ec.dtype != "bfloat16":
            raise ValueError(f"the Llama serving model runs in bfloat16, not {ec.dtype}")
        return cls(cfg, device=device, backend=backend, seed=ec.seed, num_pages=num_pages,
                   max_model_len=ec.max_model_len, fused_max_batch=ec.fused_max_batch,
                   decode_weights=ec.decode_weights, kv_cache_dtype=ec.kv_cache_dtype,
                   packed_decode=ec.packed_decode, prefill_weights=ec.prefill_weights,
                   fuse_splitk=ec.fuse_splitk, w4x_panels=ec.w4x_panels, gate_up_panels=ec.gate_up_panels)

    def __init__(self, cfg: LlamaConfig, device="cuda", backend: str = "kgs", seed: int = 0,
                 num_pages: int = 1024, max_model_len: int = 8192, fused_max_batch: int = 48,
                 decode_weights: str = "bf16", kv_cache_dtype: str = "bf16", packed_decode: bool = True,
                 prefill_weights: str = "bf16", fuse_splitk: bool = True, w4x_panels: bool = True,
                 gate_up_panels: bool = True):
        if cfg.head_dim != D.HEAD_DIM:
            raise ValueError(f"head_dim must be {D.HEAD_DIM}")
        self.cfg, self.backend, self.device = cfg, backend, torch.device(device)
        # decode projections on the four-wave kernel fuse into their neighbours:
        # split-K partials go straight to the next op (RoPE + KV write after
        # qkv, residual add + RMSNorm after o and down) instead of a reduce
        # launch, and an unsplit gate|up applies SwiGLU in its epilogue
        self.fuse_splitk = fuse_splitk and backend == "kgs"
        # split-K qkv decode layers: reduce + RoPE + KV write inside the attention
        # launch (KGS_ROPE_ATTN=1). Off by default: measured 2.9 % slower at batch
        # 256 (attention 86 -> 105 us against the 10 us rope_cache it replaces;
        # profiles/r3/decode/README.md, run r3r)
        self.rope_attn = os.environ.get("KGS_ROPE_ATTN", "0") == "1"
        base = LlamaModel(cfg, device=device, backend="torch" if backend == "ref" else "kgs", seed=seed)
        self.oracle = base  # same weights, full-recompute forward (tests)
        self.embed, self.norm = base.embed, base.norm
        self.ln1 = [L["ln1"] for L in base.layers]
        self.ln2 = [L["ln2"] for L in base.layers]
        self.w = [{n: base.layers[i][n].w for n in ("qkv", "o", "gate_up", "down")} for i in range(cfg.layers)]
        self.w_lm = base.lm_head.w
        self.packed = None
        self.fused_max_batch = fused_max_batch
        if decode_weights not in ("bf16", "fp8"):
            raise ValueError(f"decode_weights must be bf16 or fp8, got {decode_weights!r}")
        self.decode_fp8 = decode_weights == "fp8"
        if self.decode_fp8:
            self.fused_max_batch = min(fused_max_batch, 64)  # the W8A16 skinny GEMM covers M <= 64
        if backend == "kgs" and not packed_decode:
            # no prepacked decode copies (e.g. Llama-3-70B: one bf16 copy of the
            # weights is 141 GB): decode runs on the library/split-K GEMMs
            if self.decode_fp8:
                raise ValueError("decode_weights='fp8' needs the packed decode copies")
            self.fused_max_batch = 0
            D.reserve_workspace(self.device)
        elif backend == "kgs":
            f8 = self.decode_fp8
            # decode copies in skinny-GEMM fragment order; the RMSNorm weights
            # in front of qkv / gate|up / lm_head are folded into them (their
            # GEMMs apply the norm in the epilogue), gate|up is SwiGLU-packed,
            # and with bf16 weights and a bf16 cache qkv is RoPE-packed (its
            # epilogue rotates q / k and writes the KV cache)
            rope = None if f8 or kv_cache_dtype != "bf16" else (cfg.heads, cfg.kv_heads)
            self.packed = [{"qkv": D.PackedWeight(lw["qkv"], fold=self.ln1[i], fp8=f8, rope=rope),
                            "o": D.PackedWeight(lw["o"], fp8=f8),
                            "gate_up": D.PackedWeight(lw["gate_up"], swiglu=True, fold=self.ln2[i], fp8=f8),
                            "down": D.PackedWeight(lw["down"], fp8=f8)} for i, lw in enumerate(self.w)]
            self.packed_lm = D.PackedWeight(self.w_lm, fold=self.norm, fp8=f8)
            D.reserve_workspace(self.device)
        # split-K decode projections (qkv, o, down from batch 64 up, kgs.ops.decode
        # W4X_TUNED) read a third copy laid out tile-panel major, so each K-step's
        # weight block is one contiguous HBM run (PACKB): 5-6 % off the down
        # projection at batch 128/256 (profiles/r3/decode/README.md). 6.4 GB for
        # Llama-3-8B; kept only with the other decode copies
        self.w4x_panels = None
        if self.fuse_splitk and packed_decode and w4x_panels:
            from kgs.ops.gemm import pack_w4x_weight

            bns = {n: D.w4x_split_bns(*self.w[0][n].shape) for n in ("qkv", "o", "down")}
            self.w4x_panels = [{(n, bn): pack_w4x_weight(lw[n], bn) for n in bns for bn in bns[n]}
                               for lw in self.w]
        # SwiGLU tile-panel copies of gate|up (235 MB per layer and tile width,
        # 15 GB for Llama-3-8B) for the unsplit decode routes: with non-temporal
        # weight loads they read 4 % faster than row-major at batch 256 (64.9 vs
        # 68.0 us, profiles/r4/decode/README.md); batch-256 serving 18 302 ->
        # 18 442 output tok/s (profiles/r5/decode/README.md). Off:
        # gate_up_panels=False or KGS_GATEUP_PANELS=0.
        self.gate_up_panels = None
        if (self.fuse_splitk and packed_decode and gate_up_panels
                and os.environ.get("KGS_GATEUP_PANELS", "1") == "1"):
            from kgs.ops.gemm import pack_w4x_weight

            gbns = gate_up_panel_widths(*self.w[0]["gate_up"].shape)
            self.gate_up_panels = [{bn: pack_w4x_weight(lw["gate_up"], bn, swiglu=True) for bn in gbns}
                                   for lw in self.w]
        if prefill_weights not in ("bf16", "fp8"):
            raise ValueError(f"prefill_weights must be bf16 or fp8, got {prefill_weights!r}")
        self.prefill_f8 = None
        if prefill_weights == "fp8" and backend == "kgs":
            # W8A8 prefill (e4m3 weights, per-tensor scale; activations quantised per
            # row by the fused norm / SwiGLU producers): ~2x the bf16 GEMM rate on the
            # compute-bound prompt pass; decode and the oracle keep the bf16 weights
            from kgs.ops import Fp8Linear

            self.prefill_f8 = [{n: Fp8Linear(lw[n]) for n in ("qkv", "o", "gate_up", "down")} for lw in self.w]
        self.cache = D.PagedKVCache(cfg.layers, num_pages, cfg.kv_heads, self.device, dtype=kv_cache_dtype)
        self.max_model_len = max_model_len
        from kgs.ops.transformer import rope_tables

        self.cos, self.sin = rope_tables(max_model_len + 256, cfg.head_dim, cfg.rope_theta, self.device)

    # ------------------------------------------------------------------ utils
    def weight_bytes(self) -> int:
        n = sum(w.numel() for lw in self.w for w in lw.values()) + self.w_lm.numel()
        return 2 * n

    def _proj(self, x: torch.Tensor, layer: int | None, name: str, decode: bool) -> torch.Tensor:
        w = self.w_lm if layer is None else self.w[layer][name]
        if self.backend == "ref":
            return (x.float() @ w.float().T).to(torch.bfloat16)
        m = x.shape[0]
        if decode:
            n, k = w.shape
            table = D.w4x_route(m, n, k)
            rule = D.w4x_rule(m, n, k) if table is None else None
            route = table or (rule if rule is not None and rule[1] == 1 else None)
            if route is not None:
                from kgs.ops.gemm import gemm_nt_w4x

                return gemm_nt_w4x(x, w, bn=route[0], nslice=route[1], bm=route[2], stages=D.w4x_stages(route),
                                   nt_weights=D.w4x_nt(route), private=table is None)
            # slices whose sum nothing takes: the general kernel's tiles, but for small outputs of a middling K the
            # library's (us at 96 rows, the rule's slices and their sum / general / library: 1024x1024 9.5 / 7.0 / 8.3,
            # 2560x7168 18.9 / 17.7 / 20.3, 5120x5120 25.4 / 21.2 / 27.2; 1024x4096 14.5 / 11.5 / 8.9, 2048x2048 11.8 / 11.1 / 8.5)
            if rule is not None and not (n <= 2048 and 1024 < k <= 4096):
                from kgs.ops import gemm_nt

                return gemm_nt(x, w)
        if decode:
            ns = D.splitk_slices(m, w.shape[0], w.shape[1])
            if ns == 1:
                from kgs.ops import gemm_nt

                return gemm_nt(x, w)
            if ns is not None:
                from kgs.ops.gemm import gemm_nt_splitk

                return gemm_nt_splitk(x, w, ns)
        if decode and self.packed is not None and name in ("o", "down") and D.use_skinny(m, w.shape[0], w.shape[1]) and \
                not (self.decode_fp8 and m > 64):
            return D.skinny_gemm(x, self.packed[layer][name])
        # the LM head (N = 128256) from batch 128 up runs faster on the kgs
        # 256x256 GEMM than on hipBLASLt (1.09x at 128, 1.21x at 256,
        # profiles/decode_wide_gemm.jsonl); the other decode shapes do not
        if decode and (layer is not None or m < 128) and not (layer is None and head_on_small_tiles(m, *w.shape)):
            return torch.matmul(x, w.T)
        from kgs.ops import gemm_nt

        return gemm_nt(x, w)

    def _splitk_route(self, m: int, layer: int, name: str):
        """(bn, nslice) when this decode projection runs split-K on the
        four-wave kernel and its reduce can be fused into the consumer."""
        if not self.fuse_splitk:
            return None
        w = self.w[layer][name]
        r = D.w4x_route(m, w.shape[0], w.shape[1]) or D.w4x_rule(m, w.shape[0], w.shape[1])
        if r is None or r[1] < 2:
            return None
        if name in ("o", "down") and self.cfg.hidden % 2048:
            return None
        return r

    def _w4x_weight(self, layer: int, name: str, bn: int):
        """The weight a split-K four-wave projection reads: its tile-panel
        copy when there is one for ``bn``, else the row-major weight."""
        if self.w4x_panels is not None:
            p = self.w4x_panels[layer].get((name, bn))
            if p is not None:
                return p
        return self.w[layer][name]

    def _gate_up_weight(self, layer: int, bn: int):
        """gate|up as the SwiGLU four-wave kernel reads it: the SwiGLU tile-panel
        copy for ``bn`` when ``gate_up_panels`` made one, else row-major."""
        if self.gate_up_panels is not None and bn in self.gate_up_panels[layer]:
            return self.gate_up_panels[layer][bn]
        return self.w[layer]["gate_up"]

    def _swiglu_route(self, m: int):
        """The route when the decode gate|up projection runs on the four-wave kernel -- unsplit,
        SwiGLU goes into its epilogue, split (no measured entry is), into the slices' sum -- or the gate kernel (``GATE``
        wide)."""
        if not self.fuse_splitk:
            return None
        w = self.w[0]["gate_up"]
        r = D.w4x_route(m, w.shape[0], w.shape[1])
        if r is not None:
            return r if r[1] == 1 else None
        return gate_up_route(m, *w.shape)

    def _split_proj(self, x, layer: int, name: str, r, private: bool = False):
        """fp32 partial products of a projection along route ``r``, in a buffer of the call's own if
        ``private`` (prompts) and for a size without measured entries."""
        from kgs.ops.gemm import gemm_nt_w4x_partials

        w = self.w[layer][name]
        return gemm_nt_w4x_partials(x, self._w4x_weight(layer, name, r[0]), *r, nt_weights=D.w4x_nt(r),
                                    private=private or D.w4x_route(x.shape[0], *w.shape) is None)

    def _gate_up_split(self, y, layer: int, r):
        """gate|up and SwiGLU along route ``r`` of :meth:`_swiglu_route`."""
        from kgs.ops.gemm import gemm_gate, gemm_nt_w4x_splitk_swiglu, gemm_nt_w4x_swiglu

        if r[0] == GATE:
            return gemm_gate(y, self.w[layer]["gate_up"], r[2])
        if r[1] > 1:
            return gemm_nt_w4x_splitk_swiglu(y, self.w[layer]["gate_up"], r[0], r[1], r[2], nt_weights=D.w4x_nt(r), private=True)
        return gemm_nt_w4x_swiglu(y, self._gate_up_weight(layer, r[0]), bn=r[0], bm=r[2], stages=D.w4x_stages(r),
                                  nt_weights=D.w4x_nt(r))

    def _norm(self, x, d, w):
        """x += d (in place, bf16) and return rmsnorm(x) * w."""
        if self.backend == "ref":
            if d is not None:
                x.copy_((x.float() + d.float()).to(torch.bfloat16))
            return _rms_norm(x, w, self.cfg.eps)
        from kgs.ops.transformer import add_rmsnorm

        return add_rmsnorm(x, d, w, self.cfg.eps)

    def _proj_add_norm(self, a, layer: int, name: str, x, w):
        """Prompt pass: x += a @ W.T, return rmsnorm(x) * w. On kgs
        the residual add runs in the GEMM's store (EPI_ADDC) and the
        norm reads x once: bitwise the GEMM + add_rmsnorm pair, with one
        [rows, hidden] tensor fewer through HBM (profiles/r5/prefill_swiglu)."""
        if self.backend == "kgs":
            from kgs.ops.gemm import add_product_

            if add_product_(a, self.w[layer][name], x):
                return self._norm(x, None, w)
        return self._norm(x, self._proj(a, layer, name, False), w)

    def _gate_up_act(self, y, layer):
        """Prompt-pass SwiGLU MLP input: fused into the GEMM epilogue on kgs."""
        if self.backend == "kgs" and self.fuse_splitk:
            from kgs.ops.gemm import gemm_swiglu

            return gemm_swiglu(y, self.w[layer]["gate_up"])
        return self._silu_mul(self._proj(y, layer, "gate_up", False))

    def _silu_mul(self, gu):
        if self.backend == "ref":
            i = gu.shape[1] // 2
            g, u = gu[:, :i].float(), gu[:, i:].float()
            return (g * torch.sigmoid(g) * u).to(torch.bfloat16)
        from kgs.ops.transformer import silu_mul

        return silu_mul(gu)

    def _rope_cache(self, qkv, layer, positions, slots, rows=None):
        c = self.cfg
        if self.backend == "ref":
            hq = c.heads + c.kv_heads
            rot = D.ref_rope_rows(qkv, self.cos, self.sin, positions, hq)
            qkv[:, :hq * D.HEAD_DIM] = rot.to(torch.bfloat16)
            k = qkv[:, c.heads * D.HEAD_DIM:hq * D.HEAD_DIM].reshape(-1, c.kv_heads, D.HEAD_DIM)
            v = qkv[:, hq * D.HEAD_DIM:(hq + c.kv_heads) * D.HEAD_DIM].reshape(-1, c.kv_heads, D.HEAD_DIM)
            D.ref_cache_write(self.cache.layer(layer), k, v, slots)
            return
        D.rope_cache_(qkv, self.cos, self.sin, positions, slots, self.cache.layer(layer), c.heads, c.kv_heads, rows=rows)

    # ---------------------------------------------------------------- prefill
    @torch.no_grad()
    def prefill(self, tokens, positions, slots, seq_starts, seq_lens, padded_lens) -> torch.Tensor:
        """Flattened padded prompts -> logits of each sequence's last real token [S, vocab]."""
        c = self.cfg
        h, hd = c.hidden, c.head_dim
        if self.prefill_f8 is not None:
            return self._prefill_fp8(tokens, positions, slots, seq_starts, seq_lens, padded_lens)
        seqs = [(int(s), int(n), int(p), 0) for s, n, p in zip(seq_starts, seq_lens, padded_lens)]
        rows = sum(n for _, n, _, _ in seqs)
        if self._slab_prompts(rows) or self._fused_prompts(rows, len(seqs)):
            return self._prefill_fused(tokens, positions, slots, seqs)
        plan = self._prompt_rows(seqs, tokens.numel(), tokens.device)
        x, y = self._start(tokens, plan.keep)
        T.op("prefill embed+norm")
        m = x.shape[0]
        # few rows: the decode step's split tiles, whose sums the rotation, norms and gate take (one
        # prompt of 90 tokens at hidden 4096: 703 us by the general kernel and its own sums, 635 so)
        few = m <= D.W4X_RULE_MAX
        rq, ro, rd = (self._splitk_route(m, 0, n) if few else None for n in ("qkv", "o", "down"))
        rg = self._swiglu_route(m) if few else None
        if ro or rd:
            from kgs.ops.transformer import splitk_add_rmsnorm
        for i in range(c.layers):
            if rq:
                part = self._split_proj(y, i, "qkv", rq, True)
                qkv = torch.empty((m, part.shape[2]), dtype=torch.bfloat16, device=x.device)
                T.op(f"prefill L{i} qkv")
                D.rope_cache_(qkv, self.cos, self.sin, positions, slots, self.cache.layer(i), c.heads, c.kv_heads,
                              partials=part, rows=plan.rows)
            else:
                qkv = self._proj(y, i, "qkv", False)
                T.op(f"prefill L{i} qkv")
                self._rope_cache(qkv, i, positions, slots, plan.rows)
            T.op(f"prefill L{i} rope_cache")
            a = self._prefill_attention(qkv, seq_starts, seq_lens, padded_lens, plan)
            T.op(f"prefill L{i} attention")
            if ro:
                y = splitk_add_rmsnorm(self._split_proj(a, i, "o", ro, True), x, self.ln2[i], c.eps)
            else:
                y = self._proj_add_norm(a, i, "o", x, self.ln2[i])
            T.op(f"prefill L{i} o+norm")
            act = self._gate_up_split(y, i, rg) if rg else self._gate_up_act(y, i)
            T.op(f"prefill L{i} gate_up")
            nxt = self.ln1[i + 1] if i + 1 < c.layers else self.norm
            if rd:
                y = splitk_add_rmsnorm(self._split_proj(act, i, "down", rd, True), x, nxt, c.eps)
            else:
                y = self._proj_add_norm(act, i, "down", x, nxt)
            T.op(f"prefill L{i} down+norm")
        out = self._proj(y.index_select(0, plan.last), None, "lm", True)
        T.op("prefill lm_head")
        return out

    def _fused_prompts(self, rows: int, prompts: int) -> bool:
        """Whether a step of so many prompt rows takes the fused decode layer: as many as a decode step of it,
        64 at most (what its rotation takes), where its products tile: what tiles makes its norms' statistics itself, so that equal steps give equal bits. Not wider
        than the norm kernels of longer prompts."""
        if self.packed is None or self.decode_fp8 or not 0 < rows <= min(self.fused_max_batch, 64) or self.packed[0]["o"].n > 8192:
            return False
        return all(D.skinny_takes(rows, w.n, w.k, w.fp8, bool(w.rope)) for w in self.packed[0].values()) and \
            D.skinny_takes(prompts, self.packed_lm.n, self.packed_lm.k)

    def _prefill_fused(self, tokens, positions, slots, seqs) -> torch.Tensor:
        """A prompt step of few rows on the decode layers (:meth:`_fused_layers`, :meth:`_slab_layers`), without its padding:
        5 launches a layer besides the attention's (one prompt of 20 tokens, hidden 2048: 481 us by the
        split tiles, 403 so; of 30, hidden 4096: 630 and 546)."""
        plan = self._prompt_rows(seqs, tokens.numel(), tokens.device, drop=True, force=True)
        c = self.cfg
        from kgs.ops.transformer import attention_blocks

        def attend(qkv, i):
            a = torch.empty((plan.n, c.heads * c.head_dim), dtype=torch.bfloat16, device=qkv.device)
            return attention_blocks(qkv, *self._kv(qkv), plan.items, c.heads, c.kv_heads, a, merges=plan.merges, slots=plan.slots)

        if self._slab_prompts(plan.n):
            x, y, ss = self._slab_layers(tokens, positions, slots, attend, "prefill", keep=plan.keep)
            out = self._slab_head(x.index_select(0, plan.last) if y is None else y.index_select(0, plan.last), y is None,
                                  None if y is not None else ss.index_select(0, plan.last), decode=False)
            T.op("prefill-slabs lm_head")
            return out
        # counters of the step's own, cleared with its first launch: nothing is shared with a decode step on another stream
        most = max(w.n for w in (*self.packed[0].values(), self.packed_lm))
        count = torch.empty(most // 16, dtype=torch.int32, device=tokens.device)
        x, _ = self._fused_layers(tokens, positions, slots, attend, "prefill", count, keep=plan.keep, heads=plan.last.numel())
        out = D.own_gemm(x.index_select(0, plan.last), self.packed_lm, norm=True, eps=c.eps, counters=count)
        T.op("prefill-fused lm_head")
        return out

    def _prefill_fp8(self, tokens, positions, slots, seq_starts, seq_lens, padded_lens) -> torch.Tensor:
        """W8A8 prompt pass: every GEMM input is e4m3 rows with per-row scales from
        its fused producer (add_rmsnorm_fp8, silu_mul_fp8, quantize_rows_fp8);
        attention, RoPE/KV write, the residual stream and the LM head stay bf16."""
        from kgs.ops.transformer import add_rmsnorm, add_rmsnorm_fp8, quantize_rows_fp8, silu_mul_fp8

        c = self.cfg
        plan = self._prompt_rows([(int(s), int(n), int(p), 0) for s, n, p in zip(seq_starts, seq_lens, padded_lens)],
                                 tokens.numel(), tokens.device, drop=False)
        x, y = self._start(tokens, norm=False)
        y8, ys = add_rmsnorm_fp8(x, None, self.ln1[0], c.eps)
        for i in range(c.layers):
            F = self.prefill_f8[i]
            qkv = F["qkv"].forward_q(y8, ys)
            self._rope_cache(qkv, i, positions, slots)
            a8, as_ = quantize_rows_fp8(self._prefill_attention(qkv, seq_starts, seq_lens, padded_lens, plan))
            y8, ys = add_rmsnorm_fp8(x, F["o"].forward_q(a8, as_), self.ln2[i], c.eps)
            m8, ms = silu_mul_fp8(F["gate_up"].forward_q(y8, ys))
            d = F["down"].forward_q(m8, ms)
            if i + 1 < c.layers:
                y8, ys = add_rmsnorm_fp8(x, d, self.ln1[i + 1], c.eps)
            else:
                y = add_rmsnorm(x, d, self.norm, c.eps)
        return self._proj(y.index_select(0, plan.last), None, "lm", True)

    def _prompt_rows(self, seqs, total: int, device, drop: bool = True, tail: int = 0, wanted=None,
                     force: bool = False) -> "_PromptRows":
        """What a step's layers need of its prompt portions ``(first row, rows, padded rows, cached tokens
        before)`` and ``tail`` decode rows after them, ``total`` rows as given, in one copy to
        the device. ``wanted``: the portions whose last row is wanted, all by default.

        The layers run without the padding wherever that saves a 128-row tile of their products:
        no result takes anything from it (a product of fewer rows may add its K slices in another
        order, so fp32 sums and the bits after them can differ), and it is an eighth of the rows at 500 tokens a prompt (16 such
        prompts at hidden 4096: 12.85 ms with it, 10.32 without), most of them at 20; ``force``: in any
        case. Equal portions without cached tokens that need no rows dropped keep the batched
        launch."""
        import numpy as np

        ref = self.backend == "ref"
        real = sum(n for _, n, _, _ in seqs) + tail
        drop = drop and not ref and (force or -(-real // 128) < -(-total // 128))
        starts, at = [s for s, _, _, _ in seqs], 0
        if drop:
            starts = []
            for _, n, _, _ in seqs:
                starts.append(at)
                at += n
        else:
            at = total - tail
        last = [r + n - 1 for r, (_, n, _, _), w in zip(starts, seqs, wanted or [True] * len(seqs)) if w]
        parts = [np.asarray(last + list(range(at, at + tail)), np.int32)]
        past, items = [], None
        if not ref and seqs and (drop or wanted is not None or len({p for _, _, p, _ in seqs}) > 1):
            from kgs.ops.transformer import SPLIT_TILES, block_items, split_items

            blocks, k0 = [], 0
            for j, (r, (_, n, p, ctx)) in enumerate(zip(starts, seqs)):
                m = n if drop else p
                blocks.append((r, m, k0 if ctx else r, ctx, int(ctx > 0)))
                if ctx:
                    past.append((k0, k0 + ctx + m, ctx + n, j))
                    k0 += ctx + m
            items, merges, slots = block_items(blocks, at), None, 0
            if max(m + ctx for _, m, _, ctx, _ in blocks) > 64 * (SPLIT_TILES - 1):  # else no block is long enough
                items, merges, slots = split_items(items, self.cfg.heads)
            parts.append(items.reshape(-1) if merges is None else np.concatenate([items, merges]).reshape(-1))
        if drop:
            keep = np.concatenate([np.arange(s, s + n, dtype=np.int32) for s, n, _, _ in seqs] +
                                  [np.arange(total - tail, total, dtype=np.int32)])
            rows = np.full(total, -1, np.int32)
            rows[keep] = np.arange(real, dtype=np.int32)
            parts += [rows, keep]
        sizes = [p.size for p in parts]
        # items first: they are read 16 bytes at a time
        t = torch.from_numpy(np.concatenate(parts[1:2] + parts[:1] + parts[2:]))
        if device.type == "cuda":
            t = t.pin_memory().to(device, non_blocking=True)
        out = _PromptRows(at + tail, past)
        n = sizes[1] if items is not None else 0
        if items is not None:
            out.items = t[:items.size].view(-1, 4)
            if merges is not None:
                out.merges, out.slots = t[items.size:n].view(-1, 4), slots
        out.last = t[n:n + sizes[0]]
        if drop:
            out.rows, out.keep = t[n + sizes[0]:n + sizes[0] + total], t[n + sizes[0] + total:]
        return out

    def _kv(self, qkv):
        """The key and the value columns of fused QKV rows."""
        c = self.cfg
        q, n = c.heads * c.head_dim, c.kv_heads * c.head_dim
        return qkv[:, q:q + n], qkv[:, q + n:q + 2 * n]

    def _prefill_attention(self, qkv, seq_starts, seq_lens, padded_lens, plan=None):
        c = self.cfg
        hd = c.head_dim
        out = torch.empty((qkv.shape[0], c.heads * hd), dtype=torch.bfloat16, device=qkv.device)
        if plan is not None and plan.items is not None:  # unequal prompts: one launch over all their query blocks
            from kgs.ops.transformer import attention_blocks

            return attention_blocks(qkv, *self._kv(qkv), plan.items, c.heads, c.kv_heads, out, merges=plan.merges,
                                    slots=plan.slots)
        if self.backend != "ref" and len(set(int(p) for p in padded_lens)) == 1:
            # equal padded lengths, packed back to back: one batched launch
            from kgs.ops.transformer import attention_qkv

            p = int(padded_lens[0])
            attention_qkv(qkv, len(padded_lens), p, c.heads, c.kv_heads, head_dim=hd, causal=True, out=out)
            return out
        for s0, n, p in zip(seq_starts, seq_lens, padded_lens):
            s0, n, p = int(s0), int(n), int(p)
            blk = qkv[s0:s0 + p]
            if self.backend == "ref":
                q = blk[:n, :c.heads * hd].float().reshape(n, c.heads, hd).transpose(0, 1)
                k = blk[:n, c.heads * hd:(c.heads + c.kv_heads) * hd].float().reshape(n, c.kv_heads, hd).transpose(0, 1)
                v = blk[:n, (c.heads + c.kv_heads) * hd:(c.heads + 2 * c.kv_heads) * hd].float().reshape(
                    n, c.kv_heads, hd).transpose(0, 1)
                rep = c.heads // c.kv_heads
                k, v = k.repeat_interleave(rep, 0), v.repeat_interleave(rep, 0)
                o = torch.nn.functional.scaled_dot_product_attention(q, k, v, is_causal=True)
                out[s0:s0 + n] = o.transpose(0, 1).reshape(n, c.heads * hd).to(torch.bfloat16)
                out[s0 + n:s0 + p] = 0
            else:
                from kgs.ops.transformer import attention_qkv

                attention_qkv(blk, 1, p, c.heads, c.kv_heads, head_dim=hd, causal=True, out=out[s0:s0 + p])
        return out

    # ------------------------------------------------------------------ mixed
    @torch.no_grad()
    def mixed(self, tokens, positions, slots, chunks, dec_block_tables=None, dec_ctx_lens=None) -> torch.Tensor:
        """Chunked-prefill step: prompt chunks (rows first) plus decode rows in ONE
        pass through the projections. ``chunks``: per prefill sequence
        ``(row0, n, padded, ctx0, pages, last)`` -- rows ``row0 .. row0+padded``
        hold prompt positions ``ctx0 .. ctx0+n-1`` (then padding), ``pages`` its
        block table, ``last`` whether the chunk ends the prompt. Decode rows
        follow. Returns logits for the last row of every ``last`` chunk, then
        for every decode row."""
        c = self.cfg
        hd = c.head_dim
        n_pf = sum(ch[2] for ch in chunks)
        nd = tokens.numel() - n_pf
        f8 = self.prefill_f8 is not None and n_pf > 0  # W8A8 projections for the whole mixed step
        plan = self._prompt_rows([ch[:4] for ch in chunks], tokens.numel(), tokens.device, drop=not f8, tail=nd,
                                 wanted=[bool(ch[5]) for ch in chunks])
        n_pf = plan.n - nd  # prompt rows of the layers
        k2 = v2 = None
        if plan.items is not None:
            from kgs.ops.transformer import attention_blocks

            if plan.past:
                k2, v2 = torch.empty((2, plan.past[-1][1], c.kv_heads * hd), dtype=torch.bfloat16, device=tokens.device)
        tickets = self._tickets(dec_block_tables) if nd else None
        x, y = self._start(tokens, plan.keep, not f8, tickets)
        if f8:
            from kgs.ops.transformer import add_rmsnorm_fp8, quantize_rows_fp8, silu_mul_fp8

            y8, ys = add_rmsnorm_fp8(x, None, self.ln1[0], c.eps)
        for i in range(c.layers):
            qkv = self.prefill_f8[i]["qkv"].forward_q(y8, ys) if f8 else self._proj(y, i, "qkv", False)
            self._rope_cache(qkv, i, positions, slots, plan.rows)
            a = torch.empty((x.shape[0], c.heads * hd), dtype=torch.bfloat16, device=x.device)
            if plan.items is not None:
                # every chunk in one launch: keys of first chunks are their own rows, those of later
                # ones the cached rows (this step's were just written there), gathered
                for r0, r1, ctx, j in plan.past:
                    D.gather_kv_into(self.cache.layer(i), chunks[j][4], ctx, k2[r0:r1], v2[r0:r1])
                attention_blocks(qkv, *self._kv(qkv), plan.items, c.heads, c.kv_heads, a, k2, v2, merges=plan.merges,
                                 slots=plan.slots)
            else:
                for row0, n, p, ctx0, pages, _ in chunks:
                    a[row0:row0 + p] = self._chunk_attention(qkv[row0:row0 + p], i, n, p, ctx0, pages)
            if nd:
                qd = qkv[n_pf:]
                if self.backend == "ref":
                    a[n_pf:] = D.ref_paged_decode(qd, self.cache.layer(i), dec_block_tables, dec_ctx_lens, c.heads,
                                                  c.kv_heads).to(torch.bfloat16)
                else:
                    D.paged_decode_attention(qd, self.cache.layer(i), dec_block_tables, dec_ctx_lens, c.heads,
                                             c.kv_heads, out=a[n_pf:], tickets=tickets)
            nxt = self.ln1[i + 1] if i + 1 < c.layers else self.norm
            if f8:
                F = self.prefill_f8[i]
                a8, as_ = quantize_rows_fp8(a)
                y8, ys = add_rmsnorm_fp8(x, F["o"].forward_q(a8, as_), self.ln2[i], c.eps)
                m8, ms = silu_mul_fp8(F["gate_up"].forward_q(y8, ys))
                d = F["down"].forward_q(m8, ms)
                if i + 1 < c.layers:
                    y8, ys = add_rmsnorm_fp8(x, d, nxt, c.eps)
                else:
                    y = self._norm(x, d, nxt)
                continue
            y = self._proj_add_norm(a, i, "o", x, self.ln2[i])
            act = self._gate_up_act(y, i)
            y = self._proj_add_norm(act, i, "down", x, nxt)
        if plan.last.numel() == 0:
            return torch.empty((0, c.vocab), dtype=torch.bfloat16, device=x.device)
        return self._proj(y.index_select(0, plan.last), None, "lm", True)

    def _chunk_attention(self, blk, layer, n, p, ctx0, pages):
        """The plain backend's causal attention of one prompt chunk (rows = positions ctx0 ..
        ctx0+p-1, n real) over everything cached before it plus itself; padded rows out 0."""
        c = self.cfg
        hd = c.head_dim
        if ctx0 == 0:  # first chunk: the whole-prompt path
            return self._prefill_attention(blk, [0], [n], [p])
        from kgs.ops.transformer import ref_attention_chunk

        # keys/values of positions 0 .. ctx0+n-1 (this chunk's rows were just
        # written to the cache by rope_cache)
        k, v = D.gather_kv(self.cache.layer(layer), pages, ctx0 + n)
        o = torch.zeros((p, c.heads * hd), dtype=torch.bfloat16, device=blk.device)
        o[:n] = ref_attention_chunk(blk[:n], k, v, c.heads, c.kv_heads, hd).to(torch.bfloat16)
        return o

    # ----------------------------------------------------------------- decode
    @torch.no_grad()
    def decode(self, tokens, positions, slots, block_tables, ctx_lens, pages_per_split=None) -> torch.Tensor:
        """One token per sequence -> logits [B, vocab]."""
        c = self.cfg
        m = tokens.shape[0]
        if self.backend == "kgs" and m <= self.fused_max_batch or self._slabs_pay(m) or self._wide(m):
            return self._decode_fused(tokens, positions, slots, block_tables, ctx_lens, pages_per_split)
        tickets = self._tickets(block_tables)
        x, y = self._start(tokens, zero=tickets)
        m = x.shape[0]
        rq, ro, rd = (self._splitk_route(m, 0, n) for n in ("qkv", "o", "down"))  # same shapes in every layer
        rg = self._swiglu_route(m)
        if ro or rd:
            from kgs.ops.transformer import splitk_add_rmsnorm
        # split-K qkv with KGS_ROPE_ATTN=1: its reduce + RoPE + KV write run
        # inside the attention launch (one launch per layer fewer)
        fused_attn = bool(rq) and rq[1] in (2, 4, 8) and self.backend == "kgs" and self.rope_attn and \
            c.heads // c.kv_heads <= 6
        for i in range(c.layers):
            if fused_attn:
                part = self._split_proj(y, i, "qkv", rq)
                a = D.rope_paged_decode_attention(part, self.cos, self.sin, positions, slots, self.cache.layer(i),
                                                  block_tables, ctx_lens, c.heads, c.kv_heads,
                                                  pages_per_split=pages_per_split)
                T.op(f"decode L{i} qkv+rope+attention")
            elif rq:
                part = self._split_proj(y, i, "qkv", rq)
                qkv = torch.empty((m, part.shape[2]), dtype=torch.bfloat16, device=x.device)
                D.rope_cache_(qkv, self.cos, self.sin, positions, slots, self.cache.layer(i), c.heads, c.kv_heads,
                              partials=part)
                T.op(f"decode L{i} qkv+rope_cache")
            else:
                qkv = self._proj(y, i, "qkv", True)
                self._rope_cache(qkv, i, positions, slots)
                T.op(f"decode L{i} qkv+rope_cache")
            if fused_attn:
                pass
            elif self.backend == "ref":
                a = D.ref_paged_decode(qkv, self.cache.layer(i), block_tables, ctx_lens, c.heads,
                                       c.kv_heads).to(torch.bfloat16)
            else:
                a = D.paged_decode_attention(qkv, self.cache.layer(i), block_tables, ctx_lens, c.heads, c.kv_heads,
                                             pages_per_split=pages_per_split, tickets=tickets)
                T.op(f"decode L{i} attention")
            if ro:
                y = splitk_add_rmsnorm(self._split_proj(a, i, "o", ro), x, self.ln2[i], c.eps)
            else:
                y = self._norm(x, self._proj(a, i, "o", True), self.ln2[i])
            T.op(f"decode L{i} o+norm")
            if rg:
                act = self._gate_up_split(y, i, rg)
            else:
                act = self._silu_mul(self._proj(y, i, "gate_up", True))
            T.op(f"decode L{i} gate_up")
            nxt = self.ln1[i + 1] if i + 1 < c.layers else self.norm
            if rd:
                y = splitk_add_rmsnorm(self._split_proj(act, i, "down", rd), x, nxt, c.eps)
            else:
                y = self._norm(x, self._proj(act, i, "down", True), nxt)
            T.op(f"decode L{i} down+norm")
        out = self._proj(y, None, "lm", True)
        T.op("decode lm_head")
        return out

    def _decode_fused(self, tokens, positions, slots, block_tables, ctx_lens, pages_per_split):
        """Decode with every norm / SwiGLU / residual add inside the skinny GEMMs:
        5 GEMMs + RoPE/KV-write + attention per layer, no elementwise launches.
        The consuming GEMM takes the folded RMSNorm's statistic from its own input; where one cannot,
        ss_a / ss_b carry the residual rows' sums of squares between the
        producing GEMM (residual update) and the consuming one."""
        c = self.cfg
        tickets = self._tickets(block_tables)

        def attend(qkv, i):
            return D.paged_decode_attention(qkv, self.cache.layer(i), block_tables, ctx_lens, c.heads, c.kv_heads,
                                            pages_per_split=pages_per_split, tickets=tickets)

        if self._slabs_pay(tokens.shape[0]) or self._wide(tokens.shape[0]):
            x, y, ss = self._slab_layers(tokens, positions, slots, attend, "decode", tickets=tickets)
            out = self._slab_head(x if y is None else y, y is None, ss, decode=True)
            T.op("decode-slabs lm_head")
            return out
        x, ss = self._fused_layers(tokens, positions, slots, attend, "decode", None, tickets=tickets)
        out = D.own_gemm(x, self.packed_lm, norm=True, eps=c.eps) if ss is None else D.skinny_gemm(x, self.packed_lm, rms=ss, eps=c.eps)
        T.op("decode-fused lm_head")
        return out

    def _own(self, m: int, head: int) -> bool:
        """Whether the products behind a norm of ``m`` rows' fused layers, and of ``head`` rows the LM head, make its statistics themselves."""
        P = self.packed[0]
        return all(D.own_takes(r, w.n, w.k, w.fp8, bool(w.rope)) for w, r in ((P["qkv"], m), (P["gate_up"], m), (self.packed_lm, head)))

    def _slabs(self, m: int) -> bool:
        """Whether ``m`` rows take the layers of :meth:`_slab_layers`: 33 to 96 of bf16 weights and pages, where the products tile. A
        ``fused_max_batch`` of 32 and less leaves all rows above it to the split tiles."""
        if self.packed is None or self.decode_fp8 or self.backend != "kgs" or not self.fuse_splitk or self.rope_attn or \
                not 32 < min(m, self.fused_max_batch) or m > D.SLAB_ROWS:
            return False
        P, c = self.packed[0], self.cfg
        return c.hidden % 2048 == 0 and c.hidden <= 8192 and bool(P["qkv"].rope) and \
            all(D.slab_split(m, P[n].n, P[n].k) for n in ("qkv", "o", "down")) and \
            all(D.slab_rows_tiles(m, w.n, w.k) for w in (P["gate_up"], self.packed_lm))

    def _slabs_pay(self, m: int) -> bool:
        """Whether they are the better ones too: up to 48 rows, where the fused layers are slower still, always, beyond where the products' slices are short or fill the
        CUs (:func:`kgs.ops.decode.slabs_fill`; four layers 2048 wide with a feed-forward of 11008, us a step of 64 / 96 rows by four-wave tiles 363 / 378, so 420 / 495)."""
        return self._slabs(m) and (m <= 48 or all(D.slabs_fill(m, w.n, w.k) for w in (self.packed[0][n] for n in ("qkv", "o", "down"))))

    def _wide(self, m: int) -> bool:
        """Whether 97 to 128 rows take those layers, under the conditions of fewer; gate and up go by their routes on normed rows. Four
        layers, us a decode step of 97 / 128 rows by split tiles / so, contexts of 300: 2048 wide, feed-forward 8192 339, 370 / 312, 333; 4096,
        14336 636, 701 / 593, 652; 8192, 28672 1868, 1954 / 1726, 1828; Not 11008, whose slices do not fill the CUs."""
        if not D.SLAB_ROWS < m <= D.WIDE_ROWS or self.packed is None or self.decode_fp8 or self.backend != "kgs" or not self.fuse_splitk or self.rope_attn or \
                self.fused_max_batch <= 32:
            return False
        P, c = self.packed[0], self.cfg
        return c.hidden % 2048 == 0 and c.hidden <= 8192 and bool(P["qkv"].rope) and all(
            D.wide_split(m, w.n, w.k) and D.slabs_fill(D.SLAB_ROWS, w.n, w.k) for w in (P["qkv"], P["o"], P["down"]))

    def _slab_prompts(self, m: int) -> bool:
        """:meth:`_slabs_pay` for prompts, whose launches come from the host one by one: up to 48 rows, where the fused layers have 5 a layer and these 8, only
        with layers of 72 M weights and more (us, fused / here, one prompt of 40 tokens among others and alone: 2048 wide, 61 M weights 331 / 379, 423 / 436; 80 M 387 / 382,
        499 / 439; 92 M 400 / 386, 510 / 448; 4096 wide, 67 M 386 / 381, 489 / 460; 92 M 440 / 382, 544 / 472; 218 M 576 / 479, 685 / 586). So with 97 to 128 rows, of 90 M
        on: split tiles / here, four layers and one prompt of 97, 112, 128 tokens, 2048 wide 61 M 403, 401, 402 / 421, 402, 406; 73 M 402, 403, 405 / 410, 412, 404; 4096 wide
        92 M 463, 464, 464 / 440, 450, 447; 143 M 510, 505, 516 / 451, 461, 474; 218 M at 97 and 128 599, 601 / 523, 567."""
        if not (self._wide(m) if m > D.SLAB_ROWS else self._slabs_pay(m)):
            return False
        return 48 < m <= D.SLAB_ROWS or sum(w.n * w.k for w in self.packed[0].values()) >= (72_000_000 if m <= 48 else 90_000_000)

    def _slab_gate(self, m: int):
        """Gate and up of ``m`` rows of :meth:`_slab_layers`: a route of :meth:`_swiglu_route` on normed rows, or None: :func:`kgs.ops.decode.skinny_rows` on the
        residual rows, whose inputs are not rounded behind the norm. The former from 49 rows on, where the route has tile-panel weights or is the gate kernel, but of a
        short K with many strips. us at 64 / 96 rows, route / skinny_rows: 28672x4096 from panels 42.3, 44.6 / 41.1, 45.7 (from row-major weights 51.5, 53.1); by the
        gate kernel 16384x4096 30.0, 31.5 / 30.4, 31.3, 8192x2048 14.2, 13.8 / 13.3, 15.3, but 16384x2048 15.9, 17.6 / 15.1, 16.7, 11264x2048 15.3, 16.3 / 14.2, 15.8. A step of 49 /
        64 rows, contexts of 300: 4096 wide, 14336 484, 512 / 493, 522; 8192 429, 443 / 438, 451; 2048 wide, 8192 263, 276 / 259, 274; 5632 260, 269 / 260, 267; 4096 236, 245 / 239, 248."""
        if m <= 48:
            return None
        route, w = self._swiglu_route(m), self.packed[0]["gate_up"]
        if route is None or route[1] > 1:
            return None
        if route[0] == GATE:
            return None if w.n > 8192 and w.k <= 2048 else route
        return route if self.gate_up_panels is not None and route[0] in self.gate_up_panels[0] else None

    def _slab_layers(self, tokens, positions, slots, attend, kind: str, keep=None, tickets=None):
        """As :meth:`_fused_layers`, for 33 to 128 rows: products in K slices that the rotation and the residual adds sum, gate and up whole. At one
        number of rows a row's bits do not depend on the others. ``(x, y, ss)``: the residual rows, their norm where the head wants that (else None: prompts of up
        to 48 rows, decode steps also where :func:`kgs.ops.decode.head_pays`) and else their sums of squares. Four layers 4096 wide, us a step by four-wave tiles (up to 48 rows skinny) / so: one prompt of 90
        tokens 599 / 540, of 60 615 / 509, two of 36 in all 611 / 494; 2048 wide one of 60 397 / 387."""
        from kgs.ops.transformer import embed_rows, embeds, splitk_add_rmsnorm, splitk_add_squares

        c = self.cfg
        tokens, dev = tokens.to(self.embed.device), self.embed.device
        m = (tokens if keep is None else keep).numel()
        ss, y = torch.empty(m, dtype=torch.float32, device=dev), None
        if embeds(self.embed):
            if keep is not None:
                positions, slots = positions.reshape(-1).contiguous(), slots.reshape(-1).contiguous()
            x, _, positions, slots = embed_rows(self.embed, tokens, None, c.eps, keep, ss, positions, slots, () if tickets is None else (tickets,))
        else:
            if keep is not None:
                tokens, positions, slots = (t.reshape(-1)[keep.long()] for t in (tokens, positions, slots))
            x = self.embed[tokens.long()].reshape(-1, c.hidden).contiguous()
            ss.copy_(x.float().pow(2).sum(-1))
            if tickets is not None:
                tickets.zero_()
        wide = m > D.SLAB_ROWS
        gate = self._swiglu_route(m) if wide else self._slab_gate(m)
        slabs = D.wide_slabs if wide else D.skinny_slabs
        raw = m <= 48 or kind == "decode" and D.head_pays(m, self.packed_lm.n, self.packed_lm.k)
        rope = {"cos": self.cos, "sin": self.sin, "positions": positions, "slots": slots}
        for i, P in enumerate(self.packed):
            rope["cache"] = self.cache.layer(i)
            qkv = D.rope_cache_packed(slabs(x, P["qkv"]), ss, P["qkv"], c.eps, rope)
            T.op(f"{kind}-slabs L{i} qkv+rope")
            a = attend(qkv, i)
            T.op(f"{kind}-slabs L{i} attention")
            part = slabs(a, P["o"])
            if gate or wide:
                act = splitk_add_rmsnorm(part, x, self.ln2[i], c.eps)
                act = self._gate_up_split(act, i, gate) if gate else self._silu_mul(self._proj(act, i, "gate_up", True))
            else:
                act = D.skinny_rows(x, P["gate_up"], splitk_add_squares(part, x), c.eps)
            part = slabs(act, P["down"])
            if not raw and i + 1 == c.layers:
                y = splitk_add_rmsnorm(part, x, self.norm, c.eps)
            else:
                ss = splitk_add_squares(part, x)
            T.op(f"{kind}-slabs L{i} o+mlp")
        return x, y, ss

    def _slab_head(self, x, raw: bool, ss, decode: bool):
        """Logits of rows of :meth:`_slab_layers`: residual rows with their sums of squares (``raw``), or their norm."""
        if not raw:
            return self._proj(x, None, "lm", decode)
        if x.shape[0] <= 8 and D.few_takes(x.shape[0], self.packed_lm.n, self.packed_lm.k):
            return D.skinny_few(x, self.packed_lm, norm=True, eps=self.cfg.eps)
        return (D.wide_rows if x.shape[0] > D.SLAB_ROWS else D.skinny_rows)(x, self.packed_lm, ss, self.cfg.eps)

    def _tickets(self, block_tables):
        """Tickets of the step's own for the decode rows' attention, to be cleared with its first launch; None: it takes none."""
        if self.backend != "kgs":
            return None
        n = D.part_tickets(block_tables.shape[0], self.cfg.kv_heads, block_tables.shape[1], self.cache.fp8)
        return torch.empty(n, dtype=torch.int32, device=block_tables.device) if n else None

    def _start(self, tokens, keep=None, norm: bool = True, zero=None):
        """The residual rows of a step (of the rows ``keep`` of ``tokens``) and, with ``norm``, their norm for the first layer;
        ``zero`` is cleared."""
        from kgs.ops.transformer import embed_rows, embeds

        if self.backend == "kgs" and embeds(self.embed):
            return embed_rows(self.embed, tokens.to(self.embed.device), self.ln1[0] if norm else None, self.cfg.eps, keep,
                              zeros=() if zero is None else (zero,))[:2]
        if zero is not None:
            zero.zero_()
        tokens = tokens.reshape(-1) if keep is None else tokens.reshape(-1)[keep.long()]
        x = self.embed[tokens.long()].reshape(-1, self.cfg.hidden).contiguous()
        return x, self._norm(x, None, self.ln1[0]) if norm else None

    def _fused_layers(self, tokens, positions, slots, attend, kind: str, counters, keep=None, tickets=None, heads=None):
        """The residual rows after all layers and their sums of squares (None where the products make their own, :meth:`_own`; ``heads``: rows of
        the LM head, all); ``attend(qkv, layer)`` is the attention of the rotated rows, whose keys and values are in the cache. ``keep`` (int32): of
        these rows of ``tokens``, ``positions`` and ``slots`` only. ``counters`` and ``tickets``: the step's own, cleared here (not both of them)."""
        from kgs.ops.transformer import embed_rows, embeds

        c = self.cfg
        eps = c.eps
        tokens, dev = tokens.to(self.embed.device), self.embed.device
        m = (tokens if keep is None else keep).numel()
        own = self._own(m, m if heads is None else heads)
        ss = zero = None
        if not own:
            ss = torch.empty(m, dtype=torch.float32, device=dev)  # statistic for layer 0's qkv
            zero = ss_a = torch.empty_like(ss)
            ss_b = ss
        clear = tuple(t for t in (zero, counters, tickets) if t is not None)
        if embeds(self.embed):
            if keep is not None:
                positions, slots = positions.reshape(-1).contiguous(), slots.reshape(-1).contiguous()
            x, _, positions, slots = embed_rows(self.embed, tokens, None, eps, keep, ss, positions, slots, clear)
        else:
            if keep is not None:
                tokens, positions, slots = (t.reshape(-1)[keep.long()] for t in (tokens, positions, slots))
            x = self.embed[tokens.long()].reshape(-1, c.hidden).contiguous()  # residual stream
            if ss is not None:
                ss.copy_(x.float().pow(2).sum(-1))
            for t in clear:
                t.zero_()
        for i in range(c.layers):
            P = self.packed[i]
            rope = {"cos": self.cos, "sin": self.sin, "positions": positions, "slots": slots,
                    "cache": self.cache.layer(i)} if P["qkv"].rope else None
            if own:
                qkv = D.own_gemm(x, P["qkv"], norm=True, eps=eps, rope=rope, counters=counters)
            else:
                qkv = D.skinny_gemm(x, P["qkv"], rms=ss, eps=eps, counters=counters, rope=rope)
            if rope is None:
                self._rope_cache(qkv, i, positions, slots)
            T.op(f"{kind}-fused L{i} qkv+rope")
            a = attend(qkv, i)
            T.op(f"{kind}-fused L{i} attention")
            if own:
                D.own_gemm(a, P["o"], out=x, resid=True, counters=counters)
                act = D.own_gemm(x, P["gate_up"], norm=True, eps=eps, counters=counters)
                D.own_gemm(act, P["down"], out=x, resid=True, counters=counters)
            else:
                D.skinny_gemm(a, P["o"], out=x, resid_ss=ss_a, zero=ss_b, counters=counters)
                act = D.skinny_gemm(x, P["gate_up"], rms=ss_a, eps=eps, counters=counters)
                D.skinny_gemm(act, P["down"], out=x, resid_ss=ss_b, zero=ss_a, counters=counters)
                ss = ss_b
            T.op(f"{kind}-fused L{i} o+mlp")
        return x, ss
