#!/usr/bin/env python3
"""Generate acc_regs.h: MFMA / read helpers on NAMED accumulator AGPRs.

The persistent four-wave GEMM (gemm_w4p.h) keeps its 128x128 accumulator tile
in a[0:255] by name, outside the register allocator: accumulator q (the 16x16
fragment (i, n), q = 8 i + n) is a[4q : 4q+3]. Inline-asm operands cannot
compute register numbers, so every q gets its own specialisation, generated
here. Run `python native/kernels/gen_acc_regs.py` after changing it; the output
is committed.
"""
import os

HERE = os.path.dirname(os.path.abspath(__file__))
NQ = 64


def main() -> None:
    lines = [
        "// GENERATED by native/kernels/gen_acc_regs.py -- do not edit.",
        "//",
        "// Accumulator q (q = 0..63) of a wave's 128x128 fp32 tile lives in the NAMED",
        "// AGPRs a[4q : 4q+3]. The compiler never sees these values: kernels that use",
        "// this header reserve the AGPR file with KGS_ACC_RESERVE (an asm statement",
        "// clobbering a0..a255, which also makes the kernel descriptor allocate them)",
        "// and touch it only through the helpers below. This is what lets a kernel",
        "// carry the accumulators across an outer (persistent) tile loop without the",
        "// register allocator renaming them (profiles/gemm_tuning.md, 'Persistent').",
        "//",
        "//   mfma<q>(b, a)   a[4q:4q+3] += B-fragment x A-fragment (16x16x32 bf16)",
        "//   mfma0<q>(b, a)  a[4q:4q+3]  = B-fragment x A-fragment (C = 0: no reset pass)",
        "//   read<q>()       the four fp32 values, via v_accvgpr_read_b32",
        "//   zero<q>()       a[4q:4q+3] = 0",
        "//   write<q>(x)     a[4q:4q+3] = x, via v_accvgpr_write_b32 (rescales, talking.hip)",
        "//   mfma_f8<q> / mfma0_f8<q>  the same with v_mfma_f32_16x16x128_f8f6f4 (e4m3 x e4m3)",
        "// Hazards are the caller's: MFMA -> v_accvgpr_read needs the wait states the",
        "// kernels pad with s_nop before their epilogue.",
        "#pragma once",
        "",
        '#include "kgs_common.h"',
        "",
        "namespace kgs {",
        "namespace accr {",
        "",
        "template <int Q>",
        "__device__ __forceinline__ void mfma(const bf16x8& b, const bf16x8& a);",
        "template <int Q>",
        "__device__ __forceinline__ void mfma0(const bf16x8& b, const bf16x8& a);",
        "template <int Q>",
        "__device__ __forceinline__ f32x4 read();",
        "template <int Q>",
        "__device__ __forceinline__ void zero();",
        "template <int Q>",
        "__device__ __forceinline__ void write(const f32x4& x);",
        "// fp8 (OCP e4m3, A and B) 16x16x128: 32-byte operands = 8 VGPRs each",
        "typedef int i32x8 __attribute__((ext_vector_type(8)));",
        "template <int Q>",
        "__device__ __forceinline__ void mfma_f8(const i32x8& b, const i32x8& a);",
        "template <int Q>",
        "__device__ __forceinline__ void mfma0_f8(const i32x8& b, const i32x8& a);",
        "",
    ]
    for q in range(NQ):
        lo, hi = 4 * q, 4 * q + 3
        rng = f"a[{lo}:{hi}]"
        lines += [
            "template <>",
            f"__device__ __forceinline__ void mfma<{q}>(const bf16x8& b, const bf16x8& a) {{",
            f'  asm volatile("v_mfma_f32_16x16x32_bf16 {rng}, %0, %1, {rng}" ::"v"(b), "v"(a));',
            "}",
            "template <>",
            f"__device__ __forceinline__ void mfma0<{q}>(const bf16x8& b, const bf16x8& a) {{",
            f'  asm volatile("v_mfma_f32_16x16x32_bf16 {rng}, %0, %1, 0" ::"v"(b), "v"(a));',
            "}",
            "template <>",
            f"__device__ __forceinline__ f32x4 read<{q}>() {{",
            "  float x0, x1, x2, x3;",
            "  asm volatile(",
            f'      "v_accvgpr_read_b32 %0, a{lo}\\n\\tv_accvgpr_read_b32 %1, a{lo + 1}\\n\\t"',
            f'      "v_accvgpr_read_b32 %2, a{lo + 2}\\n\\tv_accvgpr_read_b32 %3, a{lo + 3}"',
            '      : "=v"(x0), "=v"(x1), "=v"(x2), "=v"(x3));',
            "  return f32x4{x0, x1, x2, x3};",
            "}",
            "template <>",
            f"__device__ __forceinline__ void mfma_f8<{q}>(const i32x8& b, const i32x8& a) {{",
            f'  asm volatile("v_mfma_f32_16x16x128_f8f6f4 {rng}, %0, %1, {rng}" ::"v"(b), "v"(a));',
            "}",
            "template <>",
            f"__device__ __forceinline__ void mfma0_f8<{q}>(const i32x8& b, const i32x8& a) {{",
            f'  asm volatile("v_mfma_f32_16x16x128_f8f6f4 {rng}, %0, %1, 0" ::"v"(b), "v"(a));',
            "}",
            "template <>",
            f"__device__ __forceinline__ void zero<{q}>() {{",
            f'  asm volatile("v_accvgpr_write_b32 a{lo}, 0\\n\\tv_accvgpr_write_b32 a{lo + 1}, 0\\n\\t"',
            f'               "v_accvgpr_write_b32 a{lo + 2}, 0\\n\\tv_accvgpr_write_b32 a{lo + 3}, 0");',
            "}",
            "template <>",
            f"__device__ __forceinline__ void write<{q}>(const f32x4& x) {{",
            f'  asm volatile("v_accvgpr_write_b32 a{lo}, %0\\n\\tv_accvgpr_write_b32 a{lo + 1}, %1\\n\\t"',
            f'               "v_accvgpr_write_b32 a{lo + 2}, %2\\n\\tv_accvgpr_write_b32 a{lo + 3}, %3" ::"v"(x[0]), "v"(x[1]),',
            '               "v"(x[2]), "v"(x[3]));',
            "}",
        ]
    clob = ", ".join(f'"a{r}"' for r in range(4 * NQ))
    half = ", ".join(f'"a{r}"' for r in range(2 * NQ))
    quarter = ", ".join(f'"a{r}"' for r in range(NQ))
    lines += [
        "",
        "}  // namespace accr",
        "}  // namespace kgs",
        "",
        "// Reserve a0..a255 for the named accumulators (see the top of this file).",
        f'#define KGS_ACC_RESERVE() asm volatile("s_nop 0" ::: {clob})',
        "// ... or only a0..a127 (accumulators 0..31)",
        f'#define KGS_ACC_RESERVE_HALF() asm volatile("s_nop 0" ::: {half})',
        "// ... or only a0..a63 (accumulators 0..15)",
        f'#define KGS_ACC_RESERVE_QUARTER() asm volatile("s_nop 0" ::: {quarter})',
        "",
    ]
    with open(os.path.join(HERE, "acc_regs.h"), "w") as f:
        f.write("\n".join(lines))


if __name__ == "__main__":
    main()
