"""Projections ``x @ w.T`` of models whose sizes are not tuned one by one.

:class:`Projection` picks the kernel by the number of rows, as
:class:`kgs.serve.model.ServingModel` does for its tuned shapes: the skinny GEMM
over a prepacked weight for small decode batches, split-K four-wave tiles for
larger ones, the 256x256 pipeline for prompts, the library GEMM for shapes the
kernels do not take. A gated projection (fused gate|up weight) applies
``act(gate) * up`` (``act``: a name or a :class:`kgs.ops.activation.Gate`) in the
epilogue where one exists. fp32 runs on the library's
true fp32 GEMM.
"""
from __future__ import annotations

import torch

from . import decode as D
from .activation import Gate

SKINNY_MAX_ROWS = 32   # untuned shapes: skinny GEMM up to here
SPLIT_MAX_SLICES = 8   # K slices whose sum is a launch of its own


class Projection:
    """``x @ w.T``, or ``act(x @ gate.T) * (x @ up.T)`` for ``gated=act`` with
    ``w = [gate; up]``. ``pack``: keep a second copy of the weight in the skinny
    GEMM's order for decode."""

    def __init__(self, w: torch.Tensor, gated=None, pack: bool = True):
        self.w, self.gated = w.contiguous(), None if gated is None else Gate.of(gated)
        if gated is not None and w.is_cuda:
            self.gated.limit_ptr(w.device)  # on the device before any hipGraph capture
        n, k = w.shape
        self.packed = None
        if pack and n % (32 if gated is not None else 16) == 0 and k % 64 == 0 and w.dtype == torch.bfloat16 and w.is_cuda:
            self.packed = D.PackedWeight(self.w, swiglu=gated is not None, act=gated or "silu")

    def __call__(self, x: torch.Tensor) -> torch.Tensor:
        w, act = self.w, self.gated
        if x.dtype != w.dtype or x.shape[1] != w.shape[1]:
            raise ValueError(f"x {tuple(x.shape)} {x.dtype} does not fit w {tuple(w.shape)} {w.dtype}")
        m, (n, k) = x.shape[0], w.shape
        if x.dtype == torch.bfloat16:
            if m <= D.SLAB_ROWS and self._reads(x):
                y = self._packed(x, m, n, k)
                if y is not None:
                    return y
            if act is not None:
                y = self._gated(x, m)
                if y is not None:
                    return y
            else:
                y = self._plain(x, m, n, k)
                if y is not None:
                    return y
        elif torch.backends.cuda.matmul.allow_tf32:
            raise RuntimeError("fp32 projections need torch.backends.cuda.matmul.allow_tf32 = False")
        y = torch.matmul(x, w.T)
        if act is None:
            return y
        from .activation import act_mul

        return act_mul(y, act)

    def _reads(self, x) -> bool:
        """Whether the kernels that read the packed weight can read ``x``: rows of 16-byte loads, not over one another, whose offsets fit 32 bits."""
        ld = x.stride(0)
        return self.packed is not None and x.is_cuda and x.dtype == torch.bfloat16 and x.stride(1) == 1 and x.shape[1] <= ld <= 1 << 23 and \
            ld % 8 == 0 and x.data_ptr() % 16 == 0

    def _packed(self, x, m, n, k):
        """The product by a kernel that reads the packed weight, or None: up to 32 rows that of few rows (:func:`kgs.ops.decode.few_route`; a gate
        and up of K off 512 where the gate kernel has few workgroups: us at 8 rows, gate kernel / so, 8192x768 5.8 / 5.6, 16384x768 6.7 / 9.2,
        13824x4864 28.8 / 35.5), :func:`kgs.ops.decode.skinny_rows` where it pays, or :func:`kgs.ops.decode.skinny_gemm` -- of K of 512, others
        slice badly (2048x11008 at 32 rows 54.9 us, by the library 26.9) --, from 33 rows on ``skinny_rows``."""
        few = m <= SKINNY_MAX_ROWS and D.few_route(m, n, k, True)
        if few and not (self.gated is not None and k % 512 and n > (8192 if m <= 8 else 4096)):
            return D.skinny_few(x, self.packed)
        if D.rows_pay(m, n, k, self.gated is not None):
            return D.skinny_rows(x, self.packed)
        return D.skinny_gemm(x, self.packed) if m <= SKINNY_MAX_ROWS and k % 512 == 0 and D.skinny_takes(m, n, k) else None

    def partials(self, x: torch.Tensor) -> torch.Tensor:
        """:meth:`__call__`, or where it pays (:func:`kgs.ops.decode.slabs_pay`) the product of a decode batch in K slices, fp32 ``[slices, M, N]``, for a
        consumer that adds them and rounds to bf16. One slice is stored as such (its sum is no work), and rows that the kernel cannot read go the other way."""
        p = self.packed
        if self.gated is not None or x.shape[1] != self.w.shape[1] or not self._reads(x) or not D.slabs_pay(x.shape[0], p.n, p.k):
            return self(x)
        return D.skinny_slabs(x, p)

    def two(self, x: torch.Tensor, other: Projection, x2: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
        """``self(x), other(x2)``: one launch where both are products of few rows of the same sizes (2048x128 twice at 1 row 3.7 us / 2.0, at 32 4.3 / 2.3)."""
        p, q, m = self.packed, other.packed, x.shape[0]
        if m <= SKINNY_MAX_ROWS and self.gated is None and other.gated is None and self.w.shape == other.w.shape and x.shape == x2.shape and \
                x.stride() == x2.stride() and x.shape[1] == self.w.shape[1] and self._reads(x) and other._reads(x2) and D.few_route(m, *self.w.shape, True):
            return D.skinny_few_two(x, p, x2, q)
        return self(x), other(x2)

    def _gated(self, x, m):
        from .gemm import gemm_gate, gemm_nt_w4x_swiglu, gemm_swiglu, swiglu_fused_ok

        if m > 512:
            return gemm_swiglu(x, self.w, self.gated)
        if not swiglu_fused_ok(x, self.w):
            return None
        # up to 128 rows one tile high, each weight read once and non-temporal; above, the general
        # kernel's tiles (us against 256-row ones here: 5120x2048 at 256 rows 22.4 / 28.1, at 512
        # 22.7 / 28.2; 22016x4096 64.2 / 63.0 and 88.7 / 110.2)
        if m > 128:
            return gemm_swiglu(x, self.w, self.gated)
        bm = D.gate_rule(m, *self.w.shape, sliced=False)
        if bm is not None:
            return gemm_gate(x, self.w, bm, self.gated)
        return gemm_nt_w4x_swiglu(x, self.w, bn=128, bm=128, nt_weights=D.NT_WEIGHTS, act=self.gated)

    def _plain(self, x, m, n, k):
        from .gemm import gemm_nt, gemm_nt_w4x

        if m > 512:
            return gemm_nt(x, self.w)
        if m < D.W4X_MIN_BATCH or x.stride(0) % 8 or x.data_ptr() % 16:
            return None
        table = D.w4x_route(m, n, k)
        route = table or D.w4x_rule(m, n, k, SPLIT_MAX_SLICES)
        if table is None and route is not None and m > 128 and k > 4096 and n <= 16384:
            # 128-row tiles read the weight twice, and the sum of slices is a launch of its own here: the
            # general kernel instead, and 256-row tiles in two slices where those nearly fill the CUs. us at
            # 129 rows, rule / general / two slices: 4096x8192 28.3 / 25.4 / -, 7168x5120 38.7 / 30.6 / -,
            # 11008x8192 74.5 / 50.4 / -, 14336x5120 60.7 / 50.5 / 48.6, 16384x8192 87.1 / 86.6 / 75.0; at
            # K = 4096 the rule's are as good or better (8192 at 256 rows 31.1 / 40.4)
            route = (128, 2, 256) if n > 12800 and k % 256 == 0 else None
        if route is None:  # us at 64 rows of 4096x11008, which slices badly: 27 here, 36 by the library
            return gemm_nt(x, self.w) if m >= 128 or (n % 128 == 0 and k % 128 == 0) else None
        return gemm_nt_w4x(x, self.w, bn=route[0], nslice=route[1], bm=route[2], stages=D.w4x_stages(route),
                           nt_weights=D.w4x_nt(route), private=table is None)
