// Skinny products of up to 64 rows in K slices, as fp32 partial sums that the next launch adds: P[slice][M][N] of
// x[M, K] . W^T, W packed as for decode.hip's skinny ([N/16][K/32][64][8]).
//
// A workgroup of four waves takes 64 R rows of W (wave w its R tiles) over one slice. W streams into registers, PF k-steps
// ahead and past the caches; x comes by LDS-DMA in MFMA operand order, chunks of KC k-steps in three stages, one barrier
// each, and a k-step's fragments are read from LDS under the MFMAs of the one before. All loads are counted by hand: the
// compiler's own schedule waits for every load in flight before it stores a chunk (twice the time).
//
// skinny adds its slices itself: each stores its part, the last one of a strip to arrive reads them all. That is 3 to 5 us at the end of a
// launch (2048x8192 at 24 rows 14.7 us, the same product here 8.8); where the next launch passes over the output anyway it
// reads a few MB instead. Workgroups by slices (slab_split): about one a CU, and wide tiles only where N alone has enough.
#include "decode_common.h"

namespace kgs {
namespace dec {

struct SlabArgs {
  const unsigned short* x;
  const unsigned short* w;
  float* p;
  int M, N, K, ldx, ns;
};

__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, void* lds, int v, int s) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (KGS_LDS void*)lds, 16, v, s, 0, 0);
}
// all but the last VM vector loads are there, and the wave's LDS reads
template <int VM, bool LDS>
__device__ __forceinline__ void wait_loads() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4) | ((LDS ? 0 : 15) << 8));
  asm volatile("" ::: "memory");
}

template <int MT, int R>
__global__ __launch_bounds__(256, 2) void slabs(SlabArgs a) {
  constexpr int KC = MT == 1 ? 4 : 2, PF = 4, XL = KC * MT / 4;  // x fragments of a wave and chunk
  __shared__ __attribute__((aligned(16))) bf16x8 xs[3][KC * MT * 64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), fr = lane & 15, fq = lane >> 4;
  const int M = a.M, N = a.N, nkk = a.K / 32, tiles = N / (64 * R), tile = blockIdx.x % tiles, sl = blockIdx.x / tiles;
  const int nsteps = nkk / a.ns, k0 = sl * nsteps, nchunks = nsteps / KC;
  const int nt0 = (tile * 4 + w) * R;
  const auto rw = rsrc(a.w + (long)nt0 * nkk * 512, (unsigned)(R * nkk * 1024));
  const auto rx = rsrc(a.x, (unsigned)(((M - 1) * a.ldx + a.K) * 2));
  const int wo = lane * 16;
  int xo[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int f = w * XL + i, kk = f / MT, c = f % MT;
    xo[i] = 2 * (min(16 * c + fr, M - 1) * a.ldx + (k0 + kk) * 32 + fq * 8);  // rows from M on repeat the last one: never stored
  }
  bf16x8 wf[PF][R], b[2][MT];
  auto load_w = [&](int p, int s) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      wf[p][r] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rw, wo, (r * nkk + k0 + s) * 1024, 2));
  };
  int next = 0, to = 0;  // chunk to send for and its stage; past the end the last one again
  auto send = [&] {
#pragma unroll
    for (int i = 0; i < XL; ++i) dma16(rx, &xs[to][(w * XL + i) * 64], xo[i], min(next, nchunks - 1) * (KC * 64));
    ++next;
    to = to == 2 ? 0 : to + 1;
  };
  f32x4v acc[R][MT];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < MT; ++c) acc[r][c] = f32x4v{0.f, 0.f, 0.f, 0.f};
  send();
  send();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int p = 0; p < PF / 2; ++p) load_w(p, p);
  __builtin_amdgcn_sched_barrier(0);
  send();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int p = PF / 2; p < PF; ++p) load_w(p, p);
  wait_loads<2 * XL + PF * R, false>();  // chunk 0
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  int from = 0;  // stage being read
#pragma unroll
  for (int c = 0; c < MT; ++c) b[0][c] = xs[0][c * 64 + lane];
  for (int s0 = 0; s0 < nsteps; s0 += PF) {
    const int s1 = min(s0 + PF, nsteps - PF);
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      const int kk = p % KC;
      if (kk == KC - 1) {
        // the next chunk: at least the weights of 2 KC - 1 k-steps and one chunk were sent for after it. Every wave has read
        // this one, so its stage is free
        wait_loads<(2 * KC - 1) * R + XL, true>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        from = from == 2 ? 0 : from + 1;
#pragma unroll
        for (int c = 0; c < MT; ++c) b[(p + 1) & 1][c] = xs[from][c * 64 + lane];
        send();
      } else {
#pragma unroll
        for (int c = 0; c < MT; ++c) b[(p + 1) & 1][c] = xs[from][((kk + 1) * MT + c) * 64 + lane];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < MT; ++c)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[p][r], b[p & 1][c], acc[r][c], 0, 0, 0);
      load_w(p, s1 + p);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the tail's chunks land before LDS is released
#pragma unroll
  for (int c = 0; c < MT; ++c) {
    const int m = 16 * c + fr;
    if (m < M) {
#pragma unroll
      for (int r = 0; r < R; ++r) *(f32x4v*)(a.p + ((long)sl * M + m) * N + 16 * (nt0 + r) + 4 * fq) = acc[r][c];
    }
  }
}

}  // namespace dec
}  // namespace kgs

// P[ns][M][N] (fp32) = the K slices' products of x[M, K] (rows ldx apart) and W^T, W packed as for kgs_skinny_gemm_bf16: up to 64
// rows, r (1, 2) tiles of 16 W rows a wave, N a multiple of 64 r, K of 128 ns.
KGS_EXPORT int kgs_skinny_slabs(const void* wp, const void* x, float* p, int M, int N, int K, long ldx, int r, int ns, hipStream_t s) {
  using namespace kgs::dec;
  if (M < 1 || M > 64 || N <= 0 || K <= 0 || (r != 1 && r != 2) || ns < 1 || N % (64 * r) || K % (128 * ns) || (long)N * K > (1l << 31))
    return KGS_ERR_SHAPE;
  if (ldx < K || ldx > 1l << 23) return KGS_ERR_SHAPE;
  if ((uintptr_t)wp % 16 || (uintptr_t)x % 16 || (uintptr_t)p % 16 || ldx % 8) return KGS_ERR_ALIGN;
  const SlabArgs a{(const unsigned short*)x, (const unsigned short*)wp, p, M, N, K, (int)ldx, ns};
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(N / (64 * r) * ns), dim3(256), 0, s, a);
    return (int)hipGetLastError();
  };
  if (M <= 16) return r == 1 ? run(slabs<1, 1>) : run(slabs<1, 2>);
  if (M <= 32) return r == 1 ? run(slabs<2, 1>) : run(slabs<2, 2>);
  return r == 1 ? run(slabs<4, 1>) : run(slabs<4, 2>);
}
