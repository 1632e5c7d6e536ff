// The elementwise half of a linear layer's backward pass in one pass over memory: the gradient
// through the activation, its transpose (the weight gradient's operand, where that product wants
// one) and the bias gradient's column sums.
//
//   gz[m, n] = bf16(gy[m, n] act'(z[m, n])),  gzt = gz^T,  gb[n] = bf16(sum over m of gz[m, n])
//
// Everything is computed in fp32 from the bf16 inputs; the sums are those of the rounded gz. Bound
// by memory. A workgroup takes 64 columns of a strip of rows: a 64x64 tile at a time, 16 bytes per lane
// on both sides, through LDS for the transpose; its column sums go to a partial row, and a second
// launch adds the partial rows (none where one strip holds all rows). A strip has 512 rows, fewer
// where that gives less than two workgroups per CU (us with 512 rows always / so: 1024 x 310 26 / 7,
// 3584 x 960 21 / 12).
//
// Columns of no multiple of 8: gz has rows of whole 16-byte chunks, zeros past N, as the products
// that follow read them (written for no activation too), and the loads are 16 bytes at 2-byte alignment.
#include "kgs_common.h"

namespace kgs {
namespace lgrad {

enum { ACT_NONE = 0, ACT_GELU = 2, ACT_RELU = 3, ACT_SILU = 4 };  // Epi's numbers
constexpr int TILE = 64, TP = 72;                                // TP: LDS pitch, 16-B rows on staggered banks

typedef short bf16x8u __attribute__((ext_vector_type(8), aligned(2)));

template <int ACT>
__device__ __forceinline__ float grad(float g, float z) {
  if constexpr (ACT == ACT_RELU) return z <= 0.f ? 0.f : g;
  if constexpr (ACT == ACT_SILU) {
    const float s = __builtin_amdgcn_rcpf(1.0f + __expf(-z));
    return g * s * (1.0f + z * (1.0f - s));
  }
  if constexpr (ACT == ACT_GELU) {
    // with s = sigmoid(2 u) from e = exp(-2 |u|): (1 + tanh u) / 2 = s, (1 - tanh^2 u) / 2 = 2 e / (1 + e)^2
    const float k0 = 0.7978845608028654f, k1 = 0.044715f, q = z * z, u = k0 * z * (1.0f + k1 * q);
    const float e = __expf(-2.0f * fabsf(u)), r = __builtin_amdgcn_rcpf(1.0f + e), er = e * r;
    return g * ((u < 0.f ? er : r) + z * (2.0f * er * r) * (k0 * (1.0f + 3.0f * k1 * q)));
  }
  return g;
}

struct Args {
  const unsigned short *gy, *z;  // [M, N]
  unsigned short *gz, *gzt;      // [M, ldz], [N, M]; null: not wanted
  float* part;                   // [strips][N]
  unsigned short* gb;            // [N]; null: no sums
  int M, N, ldz, strip;
};

// VEC: N % 8 == 0 and (with gzt) M % 8 == 0, every pointer 16-B aligned. gz: 16-B rows always
template <int ACT, bool VEC>
__global__ __launch_bounds__(256) void act_grad(Args a) {
  __shared__ __attribute__((aligned(16))) unsigned short tile[TILE * TP];
  __shared__ float sums[32][TILE + 1];
  const int t = threadIdx.x, c0 = blockIdx.x * TILE, r0 = blockIdx.y * a.strip;
  const int ch = (t & 7) * 8, gc = c0 + ch;
  const int r1 = min(a.M, r0 + a.strip);
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int rt = r0; rt < r1; rt += TILE) {
    bf16x8 g[2], z[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int r = rt + (t >> 3) + 32 * k;
      const long at = (long)r * a.N + gc;
      g[k] = z[k] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
      if (r >= r1) continue;
      if constexpr (VEC) {
        if (gc < a.N) {
          g[k] = *(const bf16x8*)(a.gy + at);
          if constexpr (ACT != ACT_NONE) z[k] = *(const bf16x8*)(a.z + at);
        }
      } else if (gc + 8 <= a.N) {
        g[k] = *(const bf16x8u*)(a.gy + at);
        if constexpr (ACT != ACT_NONE) z[k] = *(const bf16x8u*)(a.z + at);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (gc + e < a.N) {
            g[k][e] = (short)a.gy[at + e];
            if constexpr (ACT != ACT_NONE) z[k][e] = (short)a.z[at + e];
          }
      }
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int rl = (t >> 3) + 32 * k, r = rt + rl;
      if constexpr (ACT != ACT_NONE) {
        float y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = grad<ACT>(bf2f((unsigned short)g[k][e]), bf2f((unsigned short)z[k][e]));
        g[k] = pack_bf16x8(y, 0);  // 0 past N, where gy and z were taken as 0
      }
      if (a.gz && r < r1 && gc < a.N) *(bf16x8*)(a.gz + (long)r * a.ldz + gc) = g[k];
      if (r < r1) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] += bf2f((unsigned short)g[k][e]);
      }
      if (a.gzt) *(bf16x8*)&tile[rl * TP + ch] = g[k];
    }
    if (a.gzt) {
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int col = (t >> 3) + 32 * k, rb = (t & 7) * 8, oc = c0 + col, orow = rt + rb;
        bf16x8 v;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (short)tile[(rb + j) * TP + col];
        if (oc < a.N) {
          unsigned short* o = a.gzt + (long)oc * a.M + orow;
          if constexpr (VEC) {
            if (orow < a.M) *(bf16x8*)o = v;
          } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (orow + j < a.M) o[j] = (unsigned short)v[j];
          }
        }
      }
      __syncthreads();
    }
  }
  if (!a.gb) return;
#pragma unroll
  for (int e = 0; e < 8; ++e) sums[t >> 3][ch + e] = s[e];
  __syncthreads();
  if (t < TILE && c0 + t < a.N) {
    float x = 0.f;
#pragma unroll
    for (int i = 0; i < 32; ++i) x += sums[i][t];
    if (gridDim.y == 1) a.gb[c0 + t] = f2bf(x);
    else a.part[(long)blockIdx.y * a.N + c0 + t] = x;
  }
}

__global__ __launch_bounds__(256) void sum_parts(const float* __restrict__ part, unsigned short* __restrict__ gb, int N, int n) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= N) return;
  float x = 0.f;
  for (int i = 0; i < n; i += 8) {  // eight rows' loads before the first add
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = part[(long)min(i + e, n - 1) * N + c];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (i + e < n) x += v[e];
  }
  gb[c] = f2bf(x);
}

template <int ACT>
void launch(const Args& a, dim3 grid, bool vec, hipStream_t s) {
  if (vec) hipLaunchKernelGGL((act_grad<ACT, true>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((act_grad<ACT, false>), grid, dim3(256), 0, s, a);
}

// Rows of a strip: at most 512, and short enough for two workgroups per CU, in at most 64 strips
// beyond that (their partial rows are added one by one).
inline int strip_rows(int M, int N) {
  const long tiles = (N + TILE - 1) / TILE, rt = (M + TILE - 1) / TILE;
  const long want = (512 + tiles - 1) / tiles, strips = want < 1 ? 1 : want > 64 ? 64 : want;
  const int rows = (int)((rt + strips - 1) / strips) * TILE;
  return rows < 512 ? rows : 512;
}

}  // namespace lgrad
}  // namespace kgs

// Rows of partial sums that kgs_act_grad wants for M rows of N columns (1: none).
KGS_EXPORT int kgs_act_grad_parts(int M, int N) {
  if (M <= 0 || N <= 0) return 1;
  const int strip = kgs::lgrad::strip_rows(M, N);
  return (M + strip - 1) / strip;
}

// gy, z [M, N] and gzt [N, M] contiguous bf16; gz [M, ldz], ldz % 8 == 0 and at least N, 16-B aligned, its
// rows' columns past N, up to the next multiple of 8, zeroed. act: an epilogue's number, 0 (z unused).
// gz (act 0 only), gzt, gb: null where not wanted; part: fp32 [kgs_act_grad_parts][N] for gb of several strips.
KGS_EXPORT int kgs_act_grad(const void* gy, const void* z, void* gz, void* gzt, float* part, void* gb, int M, int N, int ldz,
                            int act, hipStream_t s) {
  using namespace kgs::lgrad;
  if (M <= 0 || N <= 0) return KGS_ERR_SHAPE;
  if (gz && (ldz < N || ldz % 8 || (uintptr_t)gz % 16)) return KGS_ERR_ALIGN;
  const int strip = strip_rows(M, N), strips = (M + strip - 1) / strip, tiles = (N + TILE - 1) / TILE;
  if (act != ACT_NONE && (!z || !gz)) return KGS_ERR_ARG;
  if (gb && strips > 1 && !part) return KGS_ERR_ARG;
  const uintptr_t p = (uintptr_t)gy | (uintptr_t)z | (uintptr_t)gzt;
  const bool vec = N % 8 == 0 && p % 16 == 0 && (!gzt || M % 8 == 0);
  const Args a{(const unsigned short*)gy, (const unsigned short*)z, (unsigned short*)gz, (unsigned short*)gzt, part,
               (unsigned short*)gb, M, N, ldz, strip};
  const dim3 grid((unsigned)tiles, (unsigned)strips);
  switch (act) {
    case ACT_NONE: launch<ACT_NONE>(a, grid, vec, s); break;
    case ACT_GELU: launch<ACT_GELU>(a, grid, vec, s); break;
    case ACT_RELU: launch<ACT_RELU>(a, grid, vec, s); break;
    case ACT_SILU: launch<ACT_SILU>(a, grid, vec, s); break;
    default: return KGS_ERR_ARG;
  }
  if (gb && strips > 1)
    hipLaunchKernelGGL(sum_parts, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, part, (unsigned short*)gb, N, strips);
  return (int)hipGetLastError();
}
