// Skinny products of up to 128 rows past skinny's tickets and barriers: x[M, K] . W^T, W packed as for decode.hip's skinny
// ([N/16][K/32][64][8]), in K slices as fp32 partial sums P[slice][M][N] that the next launch adds (slabs), or whole, with the
// RMSNorm and the gate of a fused layer in the epilogue (rows).
//
// A workgroup of NW waves takes 16 NW R rows of W (wave w its R tiles) over one slice; the first four of them send for x. W streams into registers, four k-steps
// ahead and past the caches; x comes by LDS-DMA, chunks of KC k-steps in three stages, one barrier
// each, and a k-step's fragments are read from LDS under the MFMAs of the one before. All loads are counted by hand: the
// compiler's own schedule waits for every load in flight before it stores a chunk (twice the time). W has to lie packed: 16 rows' pieces of 64
// bytes, straight from its rows, take half as long again.
//
// A load instruction costs by the lines that each four lanes touch: x as 8 rows of 128 bytes comes at 120 bytes a ns and CU, in MFMA operand
// order (16 rows of 64 bytes, each lane another row than the next) at 37. And the last round of W's ring sends for nothing: fetching its
// k-steps again was waited for at the launch's end. us at 24 / 96 rows, operand order and full last round / so: 2048x2048 in 8 slices 4.6, 6.7 /
// 4.0, 5.6; 3072x2048 in 4 5.4, 8.1 / 4.8, 6.5; 2048x8192 in 8 8.7, 12.1 / 8.1, 10.0; 4096x14336 in 8 20.4, 26.5 / 19.5, 24.6; whole 28672x4096 at 24 / 90 41.4, 47.7 /
// 41.0, 45.2; 16384x2048 14.3, 19.5 / 13.5, 16.6. Deeper rings (8 k-steps, 5 stages), which long sums needed before, are 2 to 5 % slower now.
//
// Slices: skinny adds its slices itself: each stores its part, the last one of a strip to arrive reads them all. That is 3 to 5 us at the end of a
// launch (2048x8192 at 32 rows 15.0 us, the same product here 8.1); where the next launch passes over the output anyway it
// reads a few MB instead. Workgroups by slices (kgs/ops/decode.py slab_split): about one a CU, and wide tiles only where N alone has enough.
// From 33 rows on these beat the four-wave tiles of gemm_w4.h too, whose weights go through LDS; us at 64 and 90 rows, those / here:
// 6144x4096 14.9, 20.2 / 12.6, 14.2; 4096x14336 25.1, 27.6 / 21.4, 24.2; whole: 28672x4096 51.6, 54.2 / 41.5, 45.2; 32000x4096 61 / 46; at 128 rows
// 2048x2048 8.3 / 6.5, 3072x2048 9.7 / 7.5, 2048x8192 13.2 / 11.9, 6144x4096 18.5 / 17.1, 4096x14336 30.1 / 26.8; whole 32000x2048 34.5 / 30.9. There x counts
// as W does: with x alone left out 16384x2048 takes 16.9 of 19.3 us, with W left out 13.1, without MFMAs or LDS reads 18.8 -- the L2s pass on x once a
// workgroup, and deeper rings give nothing. K split over the waves with rings of their own (a quarter of the LDS reads) takes as long again as
// the four-wave tiles.
#include "decode_common.h"

#include <type_traits>

namespace kgs {
int cu_count();  // gemm_bf16.hip
namespace dec {

struct SlabArgs {
  const unsigned short* x;
  const unsigned short* w;
  void* y;  // OUT_SLABS: fp32 [ns][M][N]; else bf16 rows ldy apart
  int M, N, K, ldx, ns;
  long ldy;
  const float* sq;  // RMSNorm of x's rows: their sums of squares, or null
  float inv_k, eps, limit;
  int mode;  // OUT_GATED: EPI_GELU, EPI_CLAMPED
};
enum { OUT_SLABS, OUT_ROWS, OUT_GATED };

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

// HALVES: of one slice, summed apart (halves)
template <int MT, int R, int OUT, int NW, bool HALVES = false>
__global__ __launch_bounds__(64 * NW, NW == 4 ? 2 : 1) void slabs(SlabArgs a) {
  constexpr int PF = 4, NB = 3, KC = MT == 1 ? 4 : 2, XL = KC * MT / 4;  // XL: pieces of x of a wave and chunk
  static_assert(PF % KC == 0 && PF >= (NB - 2) * KC);
  __shared__ __attribute__((aligned(16))) bf16x8 xs[NB][KC * MT * 64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), fr = lane & 15, fq = lane >> 4;
  const int M = a.M, N = a.N, nkk = a.K / 32, T = N / (16 * R), strips = (T + NW - 1) / NW, sl = blockIdx.x / strips, at = blockIdx.x % strips * NW + w;
  const int nsteps = nkk / a.ns, k0 = sl * nsteps, nchunks = nsteps / KC;
  const int nt0 = min(at, T - 1) * R, rows = at < T ? M : 0;  // waves past the last tile repeat it and store nothing
  const auto rw = rsrc(a.w + (long)nt0 * nkk * 512, (unsigned)(R * nkk * 1024));
  const auto rx = rsrc(a.x, (unsigned)(((M - 1) * a.ldx + a.K) * 2));
  const int wo = lane * 16;
  // x: piece f of a chunk is 8 rows of 64 values, row f % (2 MT) * 8 + lane / 8; a row's 16-byte chunk j lies at j ^ (row / 2 % 8), so that a
  // fragment's reads touch every bank evenly
  int xo[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int f = (w & 3) * XL + i, row = f % (2 * MT) * 8 + (lane >> 3), j = (lane & 7) ^ ((row >> 1) & 7);
    xo[i] = 2 * (min(row, M - 1) * a.ldx + k0 * 32 + f / (2 * MT) * 64 + j * 8);  // rows from M on repeat the last one: never stored
  }
  const int ro[2] = {fr * 8 + (fq ^ (fr >> 1)), fr * 8 + ((4 + fq) ^ (fr >> 1))};  // of a fragment's 16 bytes: even and odd k-steps
  bf16x8 wf[PF][R], b[2][MT];
  auto load_w = [&](int p, int s) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      wf[p][r] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rw, wo, (r * nkk + k0 + s) * 1024, 2));
  };
  typedef f32x4v Sums[R][MT];
  Sums acc;
  [[maybe_unused]] Sums first;
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < MT; ++c) acc[r][c] = first[r][c] = f32x4v{0.f, 0.f, 0.f, 0.f};
  auto product = [&](auto sends) {
    constexpr int XS = decltype(sends)::value ? XL : 0;  // a wave's DMAs a chunk
    int next = 0, to = 0;  // chunk to send for and its stage; past the end the last one again
    auto send = [&] {
#pragma unroll
      for (int i = 0; i < XS; ++i) dma16(rx, &xs[to][(w * XL + i) * 64], xo[i], min(next, nchunks - 1) * (KC * 64));
      ++next;
      to = to == NB - 1 ? 0 : to + 1;
    };
    // KC k-steps of weights at least between two chunks, as in the loop
    send();
    send();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < NB - 1; ++g) {
#pragma unroll
      for (int p = g * KC; p < (g == NB - 2 ? PF : (g + 1) * KC); ++p) load_w(p, p);
      __builtin_amdgcn_sched_barrier(0);
      if (g < NB - 2) send();
      __builtin_amdgcn_sched_barrier(0);
    }
    wait_loads<(NB - 1) * XS + PF * R, false>();  // chunk 0
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int from = 0;  // stage being read
#pragma unroll
    for (int c = 0; c < MT; ++c) b[0][c] = xs[0][c * 128 + ro[0]];
    // a round of the weights' ring; the last one sends for nothing: what it would fetch again is waited for, up to 1 us of a launch
    auto round = [&](int s0, auto more, Sums& acc) {
      constexpr bool MORE = decltype(more)::value;
#pragma unroll
      for (int p = 0; p < PF; ++p) {
        const int kk = p % KC;
        if (MORE || p + 1 < PF) {
          if (kk == KC - 1) {
            // the next chunk: at least the weights of (NB - 1) KC - 1 k-steps and NB - 2 chunks were sent for after it. Every wave has read
            // this one, so its stage is free
            wait_loads<((NB - 1) * KC - 1) * R + (NB - 2) * XS, true>();
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            from = from == NB - 1 ? 0 : from + 1;
#pragma unroll
            for (int c = 0; c < MT; ++c) b[(p + 1) & 1][c] = xs[from][c * 128 + ro[0]];
            if constexpr (MORE) send();
          } else {
#pragma unroll
            for (int c = 0; c < MT; ++c) b[(p + 1) & 1][c] = xs[from][((kk + 1) / 2 * MT + c) * 128 + ro[(kk + 1) & 1]];
          }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < MT; ++c)
#pragma unroll
          for (int r = 0; r < R; ++r) acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[p][r], b[p & 1][c], acc[r][c], 0, 0, 0);
        if constexpr (MORE) load_w(p, s0 + PF + p);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    int s0 = 0;
    if constexpr (HALVES)
      for (; 2 * s0 < nsteps; s0 += PF) round(s0, std::true_type{}, first);
    for (; s0 + PF < nsteps; s0 += PF) round(s0, std::true_type{}, acc);
    round(s0, std::false_type{}, acc);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the tail's chunks land before LDS is released
  };
  if (NW == 4 || w < 4) product(std::true_type{});
  else product(std::false_type{});
#pragma unroll
  for (int c = 0; c < MT; ++c) {
    const int m = 16 * c + fr;
    float scale = 1.f;
    if constexpr (OUT != OUT_SLABS) {
      if (a.sq) scale = rsqrtf(a.sq[min(m, M - 1)] * a.inv_k + a.eps);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const f32x4v v = HALVES ? first[r][c] + acc[r][c] : OUT == OUT_SLABS ? acc[r][c] : acc[r][c] * scale;
      const int nt = nt0 + r;
      if constexpr (OUT == OUT_SLABS) {
        if (m < rows) *(f32x4v*)((float*)a.y + ((long)sl * M + m) * N + 16 * nt + 4 * fq) = v;
      } else if constexpr (OUT == OUT_ROWS) {
        if (m < rows) *(uint2*)((unsigned short*)a.y + m * a.ldy + 16 * nt + 4 * fq) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      } else {  // a tile's gate rows in lanes 0 .. 31, their up rows in the lanes 32 on
        f32x4v u, o;
#pragma unroll
        for (int i = 0; i < 4; ++i) u[i] = lane_xor32(v[i]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[i] = (a.mode & EPI_CLAMPED) ? gate_clamped(v[i], u[i], a.limit)
                 : ((a.mode & EPI_GELU) ? gate_act<GATE_GELU>(v[i]) : gate_act<GATE_SILU>(v[i])) * u[i];
        if (m < rows && fq < 2) *(uint2*)((unsigned short*)a.y + m * a.ldy + 8 * nt + 4 * fq) = uint2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
      }
    }
  }
}

}  // namespace dec
}  // namespace kgs

namespace {
constexpr int SLAB_ROWS = 96, WIDE_ROWS = 128;

// Waves of one tile each that cut T tiles of W finer than 64 r rows a workgroup, 0: none do. As few as leave one workgroup a CU: what 128 rows leave idle is
// up to half of the CUs, and 64 rows that are more than the CUs wait for a second round. us at 24 / 64 / 90 / 128 rows by four waves / so: gated 28672x4096 (seven
// waves) 40.2, 44.7, 49.9, 55.5 / 38.7, 42.0, 46.0, 52.6, 22016x4096 (six) 34.8, 42.9, 48.7, 53.8 / 31.5, 35.0, 39.7, 47.7; 6144x4096 in 4 slices (six) 11.5, 13.7, 15.6,
// 17.6 / 11.0, 12.3, 13.7, 16.1, 5120x4096 (five) 10.6, 13.1, 14.8, 16.4 / 9.7, 11.0, 12.1, 13.2. Eight of one tile are as four of two. The slices stay: 3072x2048 in 8
// by six waves 4.8, 6.0, 7.0, 8.1, in 4 by four 5.0, 5.9, 6.6, 7.4.
inline int fine_waves(int T, int r, int ns) {
  const int cus = kgs::cu_count();
  if (r == 1 ? T / 4 * ns <= cus : T / 8 * ns > cus) return 0;
  for (int nw = 5; nw < 8; ++nw)
    if ((T + nw - 1) / nw * ns <= cus) return nw;
  return 0;
}

constexpr int SLAB_CUS = 256;  // kgs/ops/decode.py CUS

// Whether a slice's halves are summed apart: where more slices would leave one workgroup a CU and the caller takes fewer (kgs/ops/decode.py _split). A chain of
// twice the length costs the sums precision; rms error against 64 bits of unit sums, most slices / fewer, in one chain / so: 4096x4096 1.37e-7 / 1.89e-7 /
// 1.35e-7, 4096x8192 1.93e-7 / 2.74e-7 / 1.91e-7, 2048x2048 1.03e-7 / 1.32e-7 / 0.99e-7. It takes no time (4096x4096 at 64 / 128 rows 9.6, 11.7 us both).
inline bool halves(int N, int K, int r, int ns) {
  const int tiles = N / (N >= 4096 && N % 128 == 0 ? 128 : 64);
  int most = 1;
  while (most < 16 && 2 * most * tiles <= SLAB_CUS && K % (256 * most) == 0) most *= 2;
  return r == 1 && ns < most && most % ns == 0;
}

template <int OUT, int MT>
int launch_mt(const kgs::dec::SlabArgs& a, int r, hipStream_t s) {
  using namespace kgs::dec;
  const int nw = fine_waves(a.N / 16, r, a.ns);
  auto run = [&](auto kernel, int strip, int waves) {
    hipLaunchKernelGGL(kernel, dim3((a.N + strip - 1) / strip * a.ns), dim3(64 * waves), 0, s, a);
    return (int)hipGetLastError();
  };
  auto one = [&](auto apart) {
    constexpr bool H = decltype(apart)::value;
    return nw == 5 ? run(slabs<MT, 1, OUT, 5, H>, 80, 5) : nw == 6 ? run(slabs<MT, 1, OUT, 6, H>, 96, 6) : nw == 7 ? run(slabs<MT, 1, OUT, 7, H>, 112, 7)
                                                                                                         : run(slabs<MT, 1, OUT, 4, H>, 64, 4);
  };
  if constexpr (OUT == OUT_SLABS)
    if (halves(a.N, a.K, r, a.ns)) return one(std::true_type{});
  return r == 1 || nw ? one(std::false_type{}) : run(slabs<MT, 2, OUT, 4>, 128, 4);
}
template <int OUT>
int launch_slabs(const kgs::dec::SlabArgs& a, int r, hipStream_t s) {
  if (a.M <= 16) return launch_mt<OUT, 1>(a, r, s);
  if (a.M <= 32) return launch_mt<OUT, 2>(a, r, s);
  if (a.M <= 64) return launch_mt<OUT, 4>(a, r, s);
  if (a.M <= 96) return launch_mt<OUT, 6>(a, r, s);
  if constexpr (OUT != kgs::dec::OUT_GATED) return launch_mt<OUT, 8>(a, r, s);
  return KGS_ERR_SHAPE;
}

int slab_shape(int most, const void* wp, const void* x, const void* y, int M, int N, int K, long ldx, int r, int ns) {
  if (M < 1 || M > most || N <= 0 || K <= 0 || (r != 1 && r != 2) || ns < 1 || N % (64 * r) || K % (128 * ns))
    return KGS_ERR_SHAPE;
  if (ldx < K || ldx > 1l << 23) return KGS_ERR_SHAPE;  // 32-bit offsets: x's rows, and a wave's 32 rows of W, whose base has 64 bits
  return (uintptr_t)wp % 16 || (uintptr_t)x % 16 || (uintptr_t)y % 16 || ldx % 8 ? KGS_ERR_ALIGN : 0;
}
}  // namespace

namespace {
int parts(int most, const void* wp, const void* x, float* p, int M, int N, int K, long ldx, int r, int ns, hipStream_t s) {
  using namespace kgs::dec;
  const int rc = slab_shape(most, wp, x, p, M, N, K, ldx, r, ns);
  if (rc) return rc;
  const SlabArgs a{(const unsigned short*)x, (const unsigned short*)wp, p, M, N, K, (int)ldx, ns, 0, nullptr, 0.f, 0.f, 0.f, 0};
  return launch_slabs<OUT_SLABS>(a, r, s);
}
int whole(int most, const void* wp, const void* x, void* y, int M, int N, int K, long ldx, long ldy, int r, int epi, const float* sq, float eps,
          float limit, hipStream_t s) {
  using namespace kgs::dec;
  const int rc = slab_shape(most, wp, x, y, M, N, K, ldx, r, 1);
  if (rc) return rc;
  const bool gated = epi & EPI_SWIGLU;
  if (ldy < (gated ? N / 2 : N)) return KGS_ERR_SHAPE;
  if (ldy % 4) return KGS_ERR_ALIGN;
  if (epi & ~(EPI_SWIGLU | EPI_GELU | EPI_CLAMPED) || (epi && !gated)) return KGS_ERR_ARG;
  const SlabArgs a{(const unsigned short*)x, (const unsigned short*)wp, y, M, N, K, (int)ldx, 1, ldy, sq, 1.f / K, eps, limit, epi};
  return gated ? launch_slabs<OUT_GATED>(a, r, s) : launch_slabs<OUT_ROWS>(a, r, s);
}
}  // namespace

// P[ns][M][N] (fp32) = the K slices' products of x[M, K] (rows ldx apart) and W^T, W packed as for kgs_skinny_gemm_bf16: up to 96
// rows, r (1, 2) tiles of 16 W rows a wave, N a multiple of 64 r, K of 128 ns.
KGS_EXPORT int kgs_skinny_slabs(const void* wp, const void* x, float* p, int M, int N, int K, long ldx, int r, int ns, hipStream_t s) {
  return parts(SLAB_ROWS, wp, x, p, M, N, K, ldx, r, ns, s);
}

// y[M, N] (bf16, rows ldy apart) = x[M, K] . W^T as kgs_skinny_slabs in one slice; sq: of x's RMSNorm (its weight folded into W) by
// these sums of squares of its rows. epi: EPI_SWIGLU (with EPI_GELU or EPI_CLAMPED and limit): y is [M, N / 2].
KGS_EXPORT int kgs_skinny_rows(const void* wp, const void* x, void* y, int M, int N, int K, long ldx, long ldy, int r, int epi,
                               const float* sq, float eps, float limit, hipStream_t s) {
  return whole(SLAB_ROWS, wp, x, y, M, N, K, ldx, ldy, r, epi, sq, eps, limit, s);
}

// The same of up to 128 rows, without gates
KGS_EXPORT int kgs_wide_slabs(const void* wp, const void* x, float* p, int M, int N, int K, long ldx, int r, int ns, hipStream_t s) {
  return parts(WIDE_ROWS, wp, x, p, M, N, K, ldx, r, ns, s);
}
KGS_EXPORT int kgs_wide_rows(const void* wp, const void* x, void* y, int M, int N, int K, long ldx, long ldy, int r, const float* sq, float eps,
                             hipStream_t s) {
  return whole(WIDE_ROWS, wp, x, y, M, N, K, ldx, ldy, r, 0, sq, eps, 0.f, s);
}
