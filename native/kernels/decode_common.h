// What the decode products share (decode.hip, decode_few.hip, decode_slabs.hip): the page layout of the KV cache, write-through stores for
// hand-offs inside a launch, and the fused epilogues' flags and statistics.
#pragma once

#include "sums64.h"

namespace kgs {
namespace dec {

typedef float f32x4v __attribute__((ext_vector_type(4)));

constexpr int HD = 128;                // head_dim
constexpr int PAGE = 32;               // tokens per KV-cache page
constexpr int PAGE_ELEMS = PAGE * HD;  // per (page, kv head, K|V): 4096 bf16 = 8 KB

// --- KV cache page layout (per page, per kv head: K region then V region) ---
// K (token tau, dim d): S^T = K.Q^T A-fragments, 16-token halves t, k-steps ks
__host__ __device__ __forceinline__ int kv_k_index(int tau, int d) {
  const int t = tau >> 4, r = tau & 15, ks = d >> 5, g = (d >> 3) & 3, j = d & 7;
  return (((t * 4 + ks) * 64) + g * 16 + r) * 8 + j;
}
// V (token tau, dim d): O^T = V^T.P^T A-fragments, 16-dim tiles dt; the k
// (token) order within a fragment is the order S^T's accumulator hands P over:
// lane group g holds tokens {4g..4g+3} of half 0 then {16+4g..16+4g+3}.
__host__ __device__ __forceinline__ int kv_v_index(int tau, int d) {
  const int dt = d >> 4, m = d & 15, g = (tau >> 2) & 3, j = (tau & 3) + 4 * (tau >> 4);
  return ((dt * 64) + g * 16 + m) * 8 + j;
}

// over the four 16-lane rows (lanes of one column), on the permlane swaps
__device__ __forceinline__ float wmax16(float v) { return xor32_max(xor16_max(v)); }
__device__ __forceinline__ float wsum16(float v) { return xor32_sum(xor16_sum(v)); }
__device__ __forceinline__ double wsum16(double v) { return xor32_sum(xor16_sum(v)); }

// In-launch hand-offs (split-K slabs, attention split partials): producers store
// WRITE-THROUGH (sc1 buffer stores) and drain, so they need no release fence (a
// release is a buffer_wbl2 of the whole XCD L2 per wave: decode attention ran
// 8x slower with one per split); the single consumer (last arriver) takes ONE
// agent-scope acquire before reading -- without it a reader on another XCD sees
// stale lines of a reused workspace (measured: wrong merges whenever splits
// landed on different XCDs). cdna_hip_programming.md Guideline 16, recipe R1.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00020000);
}
__device__ __forceinline__ void st_sc1(__amdgpu_buffer_rsrc_t r, unsigned off, f32x4v v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, 0, 16);
}
__device__ __forceinline__ f32x4v ld_sc1(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_bit_cast(f32x4v, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 16));
}
__device__ __forceinline__ void st1_sc1(__amdgpu_buffer_rsrc_t r, unsigned off, float a) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, a), r, off, 0, 16);
}
__device__ __forceinline__ float ld1_sc1(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 16));
}
typedef unsigned u32x2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void st2_sc1(__amdgpu_buffer_rsrc_t r, unsigned off, double a) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2v, a), r, off, 0, 16);
}
__device__ __forceinline__ double ld2_sc1(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 16));
}

// Fused epilogues (runtime flags in SkinnyEpi::mode, uniform per launch):
//   EPI_SWIGLU  W is the fused gate|up weight packed so that 16-row tile t holds
//               gate rows 8t..8t+7 then up rows 8t..8t+7 (kgs/ops/decode.py
//               pack_swiglu); lane l (gate) pairs with lane l ^ 32 (up) and
//               writes silu(g) * u, so y is [M, N/2].
//   EPI_RMS     RMSNorm folded into the GEMM: x is the raw residual stream,
//               the norm weight is folded into W, and each output row m is
//               scaled by rsqrt(ss_in[m] * inv_k + eps) -- ss_in being the
//               row's sum of squares, accumulated by the producer of x.
//   EPI_RESID   residual update y[m, n] += acc (y = the residual stream, in
//               place) and ss_out[m] += sum over n of the new y^2 (fp32
//               atomics), the statistic the next EPI_RMS consumer needs.
//   ss_zero     zeroed by workgroup 0 at kernel start (the sum-of-squares
//               buffer of the previous layer boundary, already consumed).
//   EPI_SUMS_IN, EPI_SUMS_OUT
//               ss_in (ss_out, ss_zero) hold SUM_WORDS integers a row instead of a
//               float: the exact sum of the workgroups' fp32 sums of squares (add_exact),
//               so that the order in which these arrive does not show in any bit.
//   EPI_OWN     EPI_RMS by statistics that the product makes from x itself (add_squares),
//               in an order of its own.
//   EPI_ROPE    W is the fused qkv weight packed so that in every q / k head
//               16-row tile t holds dims 8t..8t+7 then 64+8t..64+8t+7
//               (kgs/ops/decode.py rope_rows): lane l pairs with lane l ^ 32,
//               rotates (rotate-half RoPE at pos[m], fp32 cos/sin tables), stores
//               the row in the original order, and writes k / v into the bf16
//               paged cache slot slot[m] -- the rope_cache launch, folded in.
// Together they remove both add_rmsnorm launches, the SwiGLU launch and the
// RoPE / KV-write launch from a decode layer (kgs/serve/model.py fused path).
enum { EPI_SWIGLU = 1, EPI_RMS = 2, EPI_RESID = 4, EPI_ROPE = 8, EPI_GELU = 16, EPI_CLAMPED = 32, EPI_SUMS_IN = 64, EPI_SUMS_OUT = 128, EPI_OWN = 256 };
struct SkinnyEpi {
  int mode;
  int zero_words;  // 4-byte words of ss_zero
  const float* ss_in;
  float* ss_out;
  float* ss_zero;
  float inv_k, eps;
  const float* wscale;  // W8: per packed row dequant scale
  float limit;          // EPI_CLAMPED
  // EPI_ROPE
  const float* cosv;
  const float* sinv;
  const int* pos;
  const int* slot;
  unsigned short* cache;  // this layer's bf16 pages [pages][HKV][2][4096]
  int H, HKV;
};

// An exact sum of non-negative floats: a value m 2^(e - 149) (24-bit m) goes, shifted by e % 32, into
// integer e / 32 of eight, whose addition does not round. 2^24 * 2^31 times 512 values fit 64 bits, so a row takes
// at most 512 of them (of 16 columns and more: SUM_MAX_N). The last integer's values stay below 2^62: bit 63
// of it says that an infinity was added, bit 62 a NaN. Integer i of row m lies at [i][m]: the rows of a
// tile add to the same integer as a rule, and so to one run of memory.
constexpr int SUM_WORDS = 8, SUM_MAX_N = 8192;
__device__ __forceinline__ void add_exact(unsigned long long* acc, int rows, float v) {
  const unsigned b = __float_as_uint(v), e = b >> 23;
  const bool odd = e >= 255;
  const unsigned m = e ? (b & 0x7fffff) | 0x800000 : b, sh = e ? e - 1 : 0;
  if (odd) atomicOr(acc + (SUM_WORDS - 1) * rows, 1ull << (b == 0x7f800000u ? 63 : 62));
  else if (m) atomicAdd(acc + (sh >> 5) * rows, (unsigned long long)m << (sh & 31));
}
// ... as a float: the integers rounded to 53 bits each, added from the smallest
__device__ __forceinline__ float exact_sum(const unsigned long long* acc, int rows) {
  unsigned long long w[SUM_WORDS];
#pragma unroll
  for (int i = 0; i < SUM_WORDS; ++i) w[i] = acc[i * rows];
  const unsigned flags = (unsigned)(w[SUM_WORDS - 1] >> 62);
  double s = 0;
#pragma unroll
  for (int i = 0; i < SUM_WORDS; ++i) s += __builtin_ldexp((double)w[i], 32 * i - 149);
  return flags ? (flags & 1 ? __builtin_nanf("") : __builtin_inff()) : (float)s;
}

}  // namespace dec
}  // namespace kgs
